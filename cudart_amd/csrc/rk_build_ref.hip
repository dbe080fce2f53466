// The reference LBVH build (CUDA_buildMeshTreeLBVH, CUDA_buildMeshTreeLBVH.cu:457-681),
// rebuilt as a device-resident pipeline for gfx950:
//   k_boxes_morton   per-face box + reference 32-bit Morton code (A6, A7)
//   radix sort       (code, face) pairs with the reference tie order (A8-A10)
//   k_split_levels   level of each adjacent-code split (A11)
//   radix sort       splits grouped by level, ascending within a level (A12)
//   k_topo_ref       the host recursion of :309-455, level-synchronous (A13, A14)
//   k_leaf_boxes     leaf boxes, one wave per leaf (A15, pass 0)
//   k_refit_ref      internal boxes with the z-extent rule (A15, passes 1..)
//   k_emit_ref       node ids and records
//   reorder          faces'[i] = faces[indices[i]] (A16)
// No step goes through the host: the reference's device->host copies
// (:428, :651) and its host recursion are gone.
#include <algorithm>

#include "rk_device.h"
#include "rk_sort.h"

rk_status rk_sort_general_impl(hipStream_t st, uint32_t* keys, uint32_t* indices, uint32_t length,
                               uint32_t bit_depth, int init_indices, void* ws, size_t ws_bytes, uint32_t* err);

namespace {

using rk::Box;
using rk::Node;

__device__ __forceinline__ Box face_box(const uint4* __restrict__ faces, const float4* __restrict__ verts, uint32_t k) {
  uint4 f = faces[k];
  float4 v0 = verts[f.x], v1 = verts[f.y], v2 = verts[f.z];
  Box b;  // CUDA_calcMeshBoxes.cu:53-55: reset(v0), merge(v1), merge(v2)
  b.mn = rk::min4(rk::min4(v0, v1), v2);
  b.mx = rk::max4(rk::max4(v0, v1), v2);
  return b;
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {  // bit k -> bit 3k, k < 10
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}
__device__ __forceinline__ uint64_t spread21(uint64_t v) {  // bit k -> bit 3k, k < 21
  v &= 0x1FFFFFull;
  v = (v | (v << 32)) & 0x1F00000000FFFFull;
  v = (v | (v << 16)) & 0x1F0000FF0000FFull;
  v = (v | (v << 8)) & 0x100F00F00F00F00Full;
  v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
  v = (v | (v << 2)) & 0x1249249249249249ull;
  return v;
}

// kernel_calcMortonCodes, CUDA_buildMeshTreeLBVH.cu:115-173.
__device__ __forceinline__ uint32_t morton_ref32(const Box& b, float4 rmin, float4 rmax) {
  float4 len = rk::sub4(rmax, rmin);
  float sx = 2047.0f / len.x, sy = 2047.0f / len.y, sz = 1023.0f / len.z;
  float4 c = rk::muls4(rk::add4(b.mn, b.mx), 0.5f);
  uint32_t cx = rk::f2u_sat((c.x - rmin.x) * sx);
  uint32_t cy = rk::f2u_sat((c.y - rmin.y) * sy);
  uint32_t cz = rk::f2u_sat((c.z - rmin.z) * sz);
  // y bit k -> 3k, x bit k -> 3k+1 (k <= 10), z bit k -> 3k+2 (k <= 9); bit 10
  // of y and x land on bits 30 and 31.
  return spread10(cy) | (spread10(cx) << 1) | (spread10(cz) << 2) | (((cy >> 10) & 1u) << 30) |
         (((cx >> 10) & 1u) << 31);
}
// 30- and 63-bit codes (no reference counterpart): q = min((uint)((c-min)*(2^b/len)), 2^b-1),
// x in the highest bit of each triple.
__device__ __forceinline__ uint32_t morton30(const Box& b, float4 rmin, float4 rmax) {
  float4 len = rk::sub4(rmax, rmin);
  float sx = 1024.0f / len.x, sy = 1024.0f / len.y, sz = 1024.0f / len.z;
  float4 c = rk::muls4(rk::add4(b.mn, b.mx), 0.5f);
  uint32_t qx = min(rk::f2u_sat((c.x - rmin.x) * sx), 1023u);
  uint32_t qy = min(rk::f2u_sat((c.y - rmin.y) * sy), 1023u);
  uint32_t qz = min(rk::f2u_sat((c.z - rmin.z) * sz), 1023u);
  return (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz);
}
__device__ __forceinline__ uint64_t morton63(const Box& b, float4 rmin, float4 rmax) {
  float4 len = rk::sub4(rmax, rmin);
  float sx = 2097152.0f / len.x, sy = 2097152.0f / len.y, sz = 2097152.0f / len.z;
  float4 c = rk::muls4(rk::add4(b.mn, b.mx), 0.5f);
  uint32_t qx = min(rk::f2u_sat((c.x - rmin.x) * sx), 2097151u);
  uint32_t qy = min(rk::f2u_sat((c.y - rmin.y) * sy), 2097151u);
  uint32_t qz = min(rk::f2u_sat((c.z - rmin.z) * sz), 2097151u);
  return (spread21(qx) << 2) | (spread21(qy) << 1) | spread21(qz);
}

__global__ __launch_bounds__(256) void k_calc_boxes(const uint4* __restrict__ faces, const float4* __restrict__ verts,
                                                    uint32_t n, Box* __restrict__ boxes, uint32_t* __restrict__ indices) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  Box b = face_box(faces, verts, k);
  float4* o = reinterpret_cast<float4*>(boxes + k);
  o[0] = b.mn;
  o[1] = b.mx;
  indices[k] = k;
}

// Boxes, indices and reference codes of the faces, per * kBoxThreads per workgroup.
// counts (may be NULL): the sort's digit counts, zero already. copy (may be
// NULL): receives the faces as they are, for the reorder at the end.
constexpr uint32_t kBoxThreads = 1024;
__global__ __launch_bounds__(kBoxThreads) void k_boxes_morton32(const uint4* __restrict__ faces,
                                                                const float4* __restrict__ verts, uint32_t n,
                                                                float4 rmin, float4 rmax, Box* __restrict__ boxes,
                                                                uint32_t* __restrict__ indices,
                                                                uint32_t* __restrict__ codes, uint32_t per,
                                                                uint32_t* __restrict__ counts, uint32_t copies,
                                                                uint4* __restrict__ copy) {
  __shared__ uint32_t s_hist[4 * 256];
  s_hist[threadIdx.x] = 0u;
  __syncthreads();
  for (uint32_t u = 0; u < per; ++u) {
    const size_t kk = ((size_t)blockIdx.x * per + u) * kBoxThreads + threadIdx.x;
    if (kk >= n) break;
    const uint32_t k = (uint32_t)kk;
    const uint4 f = faces[k];
    if (copy) copy[k] = f;
    const float4 v0 = verts[f.x], v1 = verts[f.y], v2 = verts[f.z];
    Box b;  // CUDA_calcMeshBoxes.cu:53-55: reset(v0), merge(v1), merge(v2)
    b.mn = rk::min4(rk::min4(v0, v1), v2);
    b.mx = rk::max4(rk::max4(v0, v1), v2);
    float4* o = reinterpret_cast<float4*>(boxes + k);
    o[0] = b.mn;
    o[1] = b.mx;
    indices[k] = k;
    const uint32_t code = morton_ref32(b, rmin, rmax);
    codes[k] = code;
    if (counts) rk_count_digits<uint32_t, 4>(s_hist, code);
  }
  if (counts) {
    __syncthreads();
    rk_flush_digits<4, (int)kBoxThreads>(s_hist, counts, copies);
  }
}

// Zeroes the build's info words and level counts, and three runs of words.
__global__ __launch_bounds__(256) void k_lbvh_clear(uint32_t* __restrict__ info, uint32_t* __restrict__ level_count,
                                                    uint32_t* __restrict__ a, size_t na, uint32_t* __restrict__ b,
                                                    size_t nb, uint32_t* __restrict__ c, size_t nc) {
  const size_t stride = (size_t)gridDim.x * 256, t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t < RK_INFO_WORDS) info[t] = 0u;
  if (t < 64) level_count[t] = 0u;
  for (size_t i = t; i < na; i += stride) a[i] = 0u;
  for (size_t i = t; i < nb; i += stride) b[i] = 0u;
  for (size_t i = t; i < nc; i += stride) c[i] = 0u;
}

__global__ __launch_bounds__(256) void k_morton(const Box* __restrict__ boxes, uint32_t n, float4 rmin, float4 rmax,
                                                int mode, void* __restrict__ codes) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  Box b = rk::load_box(boxes + k);
  if (mode == RK_MORTON_REF32) static_cast<uint32_t*>(codes)[k] = morton_ref32(b, rmin, rmax);
  else if (mode == RK_MORTON_30) static_cast<uint32_t*>(codes)[k] = morton30(b, rmin, rmax);
  else static_cast<uint64_t*>(codes)[k] = morton63(b, rmin, rmax);
}

// kernel_findSplits, CUDA_buildMeshTreeLBVH.cu:175-233: for adjacent sorted
// codes with code[s]^code[s+1] != 0, level = clz (0 = bit 31). Here every
// position gets a key (32 = no split) so one stable 8-bit pass groups the
// splits by level, ascending within a level.
// Counts the levels as it goes, into the sort's digit counts when it takes
// them, else into level_count (counts, copies, 256 words per copy). Few
// workgroups, since each adds its counts to the same words: with 245 of 256
// threads those atomics took 5 us of 9.8 on 1M codes.
constexpr uint32_t kSplitPer = 16, kSplitThreads = 1024;  // positions per thread
__global__ __launch_bounds__(kSplitThreads) void k_split_levels(const uint32_t* __restrict__ codes, uint32_t n,
                                                                uint32_t* __restrict__ lev,
                                                                uint32_t* __restrict__ pos,
                                                                uint32_t* __restrict__ counts, uint32_t copies) {
  constexpr uint32_t kCopies = 16;  // most splits share a few levels: lanes count into copies
  __shared__ uint32_t s_count[kCopies][33];
  for (uint32_t i = threadIdx.x; i < kCopies * 33; i += kSplitThreads) (&s_count[0][0])[i] = 0u;
  __syncthreads();
#pragma unroll 4
  for (uint32_t u = 0; u < kSplitPer; ++u) {
    const uint32_t s = (blockIdx.x * kSplitPer + u) * kSplitThreads + threadIdx.x;
    if (s + 1 < n) {
      uint32_t diff = codes[s] ^ codes[s + 1];
      uint32_t level = diff ? (uint32_t)__clz((int)diff) : 32u;
      lev[s] = level;
      pos[s] = s + 1;
      atomicAdd(&s_count[threadIdx.x % kCopies][level], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x < 33) {
    uint32_t c = 0;
    for (uint32_t i = 0; i < kCopies; ++i) c += s_count[i][threadIdx.x];
    if (c) atomicAdd(&counts[(size_t)(blockIdx.x % copies) * 256 + threadIdx.x], c);
  }
}

constexpr uint32_t kTopoThreads = 1024;
constexpr uint32_t kMaxLevels = 96;
constexpr uint32_t kTopoFront = 5120;   // records of a level kept in LDS
constexpr uint32_t kTopoLists = 16384;  // splits kept in LDS
constexpr uint32_t kMedian = 0x80000000u;  // in rb: a median-split subtree
constexpr uint8_t kInternal = 1u;          // in rmeta; the left turns on the path from the root above it

// The tree's records, level by level, each level in ascending range order; a
// node's children are records rchild and rchild + 1.
struct TopoWs {
  uint32_t* ra;         // range start (sorted position)
  uint32_t* rb;         // range end
  uint32_t* rchild;
  uint8_t* rmeta;
  float* rbox;          // six per record
  uint32_t* lev_begin;  // kMaxLevels + 1 record offsets
  uint32_t* bits;       // a bit per position: a node splits there
  uint32_t* ranks;      // per kRankWords words, the bits before them
  uint32_t cap;
};
constexpr uint32_t kRankWords = 16;

// A barrier for what goes through LDS: stores to memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The first of A[lo, hi) (ascending) above a, or hi.
__device__ __forceinline__ uint32_t upper_bound(const uint32_t* A, uint32_t lo, uint32_t hi, uint32_t a) {
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (A[mid] <= a) lo = mid + 1u;
    else hi = mid;
  }
  return lo;
}

// Where the reference's level-L split pointer stops when every level-L split
// is <= a: it walks on through the (ascending) lists of levels L+1, L+2, ...
// and stops at the first entry > a (CUDA_buildMeshTreeLBVH.cu:381-392). That
// entry's list: [lo, hi), or [S, S) past them all. s_last: each list's last
// entry (0: empty list).
__device__ __forceinline__ void chain_list(const uint32_t* s_idx, const uint32_t* s_last, uint32_t L, uint32_t a,
                                           uint32_t S, uint32_t& lo, uint32_t& hi) {
  for (uint32_t k = L + 1; k < 32; ++k) {
    if (s_last[k] > a) {
      lo = s_idx[k];
      hi = s_idx[k + 1];
      return;
    }
  }
  lo = hi = S;
}

// The first of P[lo, hi) (ascending) above a, or hi, by a whole wave.
__device__ __forceinline__ uint32_t wave_upper_bound(const uint32_t* P, uint32_t lo, uint32_t hi, uint32_t a,
                                                     uint32_t lane) {
  while (hi - lo > 64u) {
    const uint32_t step = (hi - lo + 63u) / 64u, i = lo + lane * step;
    const uint32_t c = (uint32_t)__popcll(__ballot(i < hi && P[i] <= a));
    if (lo + c * step < hi) hi = lo + c * step;
    if (c) lo += (c - 1u) * step + 1u;
  }
  return lo + (uint32_t)__popcll(__ballot(lo + lane < hi && P[lo + lane] <= a));
}

__device__ __forceinline__ uint32_t block_excl_scan1024(uint32_t v, uint32_t* s_tmp /*16*/, uint32_t* total) {
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(incl, off, 64);
    if (lane >= (uint32_t)off) incl += y;
  }
  if (lane == 63) s_tmp[wave] = incl;
  lds_barrier();
  uint32_t wprefix = 0, tot = 0;
  for (uint32_t w = 0; w < kTopoThreads / 64; ++w) {
    uint32_t c = s_tmp[w];
    wprefix += (w < wave) ? c : 0u;
    tot += c;
  }
  lds_barrier();
  *total = tot;
  return wprefix + incl - v;
}

// The reference topology (createNode/createLeaf, CUDA_buildMeshTreeLBVH.cu:309-455),
// one workgroup, level by level. Nodes of a level are kept in ascending range
// order, which is the order the reference's depth-first recursion visits them,
// so the state of each level's split pointer is a function of the range start:
//  - a node with a level-L split > a (prefix of the level) stops at the first
//    one; it splits there if that split is < b;
//  - for the remaining nodes (suffix) the pointer has left level L: the first
//    such node walks into the deeper lists (chain_list); if it stops exactly at
//    the start of level L+1's list, every later suffix node meets the entry test
//    ptr == idx[L+1] (:375) and is a leaf; otherwise each later node stops at
//    chain_list(a).
// What bounds it is the chain from level to level on one CU, so the chain runs
// in LDS: the first kTopoLists splits (the lists of the top levels, which hold
// at most 2^L), and the current and the next level's records; memory is read for
// what lies beyond, and written without waiting. One node per
// lane and no work in waves without one: instruction issue is most of a level
// (with 2 and 4 nodes per lane, searches interleaved, 76 and 104 us). Depth-12 tree of 1M faces: 154 us through memory, with
// subtree counts up and down the levels for the node ids (k_emit_ref's ranks
// now); 59 us so.
__global__ __launch_bounds__(1024) void k_topo_ref(const uint32_t* __restrict__ A,
                                                   const uint32_t* __restrict__ counts, uint32_t copies, uint32_t n,
                                                   uint32_t d, int complete, TopoWs w, uint32_t* __restrict__ info) {
  __shared__ uint32_t s_list[kTopoLists];
  __shared__ uint32_t s_a[2][kTopoFront], s_b[2][kTopoFront];
  __shared__ uint8_t s_meta[2][kTopoFront];
  __shared__ uint32_t s_idx[34], s_cnt[33], s_last[33];
  __shared__ uint32_t s_lev[kMaxLevels + 2];
  __shared__ __attribute__((aligned(16))) uint32_t s_sum[2][kTopoThreads / 64];
  __shared__ uint32_t s_j0, s_flags;
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < kTopoLists && i + 1 < n; i += kTopoThreads) s_list[i] = A[i];
  if (tid < 64) {
    uint32_t c = 0;
    if (tid < 33)
      for (uint32_t k = 0; k < copies; ++k) c += counts[(size_t)k * 256 + tid];
    uint32_t incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, 64);
      if (tid >= (uint32_t)off) incl += y;
    }
    if (tid < 33) {
      s_cnt[tid] = c;
      s_idx[tid + 1] = incl;
      s_last[tid] = tid < 32 && c ? A[incl - 1] : 0u;
    }
  }
  if (tid == 0) {
    s_idx[0] = 0;
    s_flags = 0;
    s_j0 = 0xFFFFFFFFu;
    s_a[0][0] = 0;
    s_b[0][0] = n;
    s_meta[0][0] = 0;
    s_lev[0] = 0;
  }
  __syncthreads();
  const uint32_t S = s_idx[32];
  const uint32_t past_depth = s_idx[d + 1 < 33 ? d + 1 : 32];
  const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t cur = 0, end = 1, L = 0, leaves = 0, turn = 0;
  while (cur < end) {
    if (L >= kMaxLevels) {
      if (tid == 0) s_flags |= 0x80000000u;
      break;
    }
    const uint32_t now = L & 1u, next = now ^ 1u;
    const uint32_t cntL = L < 32 ? s_cnt[L] : 0u;
    const uint32_t EL = L < 32 ? s_idx[L + 1] : S;
    const uint32_t lastA = cntL ? s_last[L] : 0u;
    uint32_t j0 = 0xFFFFFFFFu;  // the first node whose walk leaves the level's list
    if (cntL != 0u && L < d) {
      for (uint32_t base = cur + wave * 64u; base < end; base += kTopoThreads) {
        const uint32_t r = base + lane, i = r - cur;
        bool leaves_list = false;
        if (r < end) {
          const uint32_t a = i < kTopoFront ? s_a[now][i] : w.ra[r], b = i < kTopoFront ? s_b[now][i] : w.rb[r];
          leaves_list = !(b & kMedian) && b - a >= 16 && a >= lastA;
        }
        const unsigned long long m = __ballot(leaves_list);
        if (m) {
          if (lane == 0) atomicMin(&s_j0, base + (uint32_t)__builtin_ctzll(m));
          break;
        }
      }
      lds_barrier();
      j0 = s_j0;
    }
    uint32_t out = end;
    for (uint32_t chunk = cur; chunk < end; chunk += kTopoThreads) {
      const uint32_t w0 = chunk + wave * 64u, r = w0 + lane;
      uint32_t a = 0, b = 0, meta = 0, split = 0, before = 0, mine = 0;
      bool median = false, internal = false;
      if (w0 < end) {  // a wave without records leaves its SIMD to the others
        if (r < end) {
          const uint32_t i = r - cur;
          if (i < kTopoFront) {
            a = s_a[now][i];
            b = s_b[now][i];
            meta = s_meta[now][i];
            w.ra[r] = a;
            w.rb[r] = b;
          } else {
            a = w.ra[r];
            b = w.rb[r];
            meta = w.rmeta[r];
          }
          median = (b & kMedian) != 0u;
          b &= ~kMedian;
        }
        const uint32_t size = b - a;  // 0 past the end: a leaf
        if (cntL != 0u && L < d) {    // createNode(split), :360-411
          uint32_t q0 = S;
          if (j0 < w0 + 64u) {  // where the walk that leaves the list stops
            const uint32_t j = j0 - cur, aj = j < kTopoFront ? s_a[now][j] : w.ra[j0];
            uint32_t l, h;
            chain_list(s_idx, s_last, L, aj, S, l, h);
            q0 = wave_upper_bound(h <= kTopoLists ? s_list : A, l, h, aj, lane);
          }
          bool search = !median && size >= 16u;
          uint32_t lo = s_idx[L], hi = EL;
          if (search && a >= lastA) {
            if (r == j0) lo = hi = q0;
            else if (q0 == EL) search = false;  // the entry test (:375): a leaf
            else chain_list(s_idx, s_last, L, a, S, lo, hi);
          }
          if (search) {
            const uint32_t q = __any(lo < hi && hi > kTopoLists) ? upper_bound(A, lo, hi, a) : upper_bound(s_list, lo, hi, a);
            if (q >= S) {
              atomicOr(&s_flags, (uint32_t)RK_FLAG_WALK_PAST_END);
            } else {
              if (q >= past_depth) atomicOr(&s_flags, (uint32_t)RK_FLAG_WALK_PAST_DEPTH);
              split = q < kTopoLists ? s_list[q] : A[q];
              internal = split < b;
            }
          }
        }
        // createNode(median), :314-339; createLeaf, :341-358: a complete tree
        // splits oversized leaves at the median
        if (!internal && (median ? size >= 224u : complete && size > 224u)) {
          internal = median = true;
          split = (a + b) >> 1;
        }
        const unsigned long long m = __ballot(internal);
        before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        mine = (uint32_t)__popcll(m);
        if (r < end) w.rmeta[r] = (uint8_t)(meta | (internal ? kInternal : 0u));
      }
      if (lane == 0) s_sum[turn][wave] = mine;
      lds_barrier();
      uint32_t total = 0, first = 0;
#pragma unroll
      for (uint32_t k = 0; k < kTopoThreads / 64; ++k) {
        const uint32_t c = s_sum[turn][k];
        first += k < wave ? c : 0u;
        total += c;
      }
      turn ^= 1u;
      if (internal) {
        const uint32_t pos = out + 2u * (first + before), i = pos - end;
        if (pos + 2 <= w.cap) {
          const uint32_t kind = median ? kMedian : 0u;
          w.rchild[r] = pos;
          if (i + 1 < kTopoFront) {  // i is even: both or neither
            s_a[next][i] = a;
            s_b[next][i] = split | kind;
            s_meta[next][i] = (uint8_t)(meta + 2u);  // one more left turn
            s_a[next][i + 1] = split;
            s_b[next][i + 1] = b | kind;
            s_meta[next][i + 1] = (uint8_t)meta;
          } else {
            w.ra[pos] = a;
            w.rb[pos] = split | kind;
            w.rmeta[pos] = (uint8_t)(meta + 2u);
            w.ra[pos + 1] = split;
            w.rb[pos + 1] = b | kind;
            w.rmeta[pos + 1] = (uint8_t)meta;
          }
          atomicOr(&w.bits[split >> 5], 1u << (split & 31u));
        } else {
          atomicOr(&s_flags, 0x40000000u);
        }
      }
      out += 2u * total;
    }
    leaves += end - cur - (out - end) / 2u;
    cur = end;
    end = out < w.cap ? out : w.cap;
    ++L;
    if (tid == 0) {
      s_lev[L] = cur;
      s_j0 = 0xFFFFFFFFu;
    }
    if (end - cur > kTopoFront) __syncthreads();
    else lds_barrier();
  }
  const uint32_t nlev = L;
  const uint32_t R = end;
  if (tid == 0) s_lev[nlev] = R;
  __syncthreads();
  for (uint32_t k = tid; k <= nlev; k += kTopoThreads) w.lev_begin[k] = s_lev[k];
  if (tid == 0) {
    uint32_t flags = s_flags & 0xFFFFu;
    if (R > n) flags |= RK_FLAG_NODES_GT_N;
    // The reference's kernel_bitonicMerge2x writes past the end of its input
    // (CUDA_bitonicSortGeneral.cu:254, CUDA_bitonicSort.cu:196) when the last
    // pair of 128-bins is partial: in the Morton sort (512 < n <= 32768) and
    // in the per-level value sorts of levels 1..d (128 < count <= 32768).
    auto merge2x_oob = [](uint32_t c) { return ((c + 127) / 128) % 2 == 0 && (c % 128) != 0; };
    if (n > 512 && n <= 32768 && merge2x_oob(n)) flags |= RK_FLAG_MERGE2X_OOB;
    for (uint32_t k = 1; k <= d; ++k) {
      uint32_t c = s_cnt[k];
      if (c > 128 && c <= 32768 && merge2x_oob(c)) flags |= RK_FLAG_MERGE2X_OOB;
    }
    info[RK_INFO_NODE_COUNT] = R;
    info[RK_INFO_REAL_DEPTH] = nlev;  // the last level is all leaves
    atomicOr(&info[RK_INFO_FLAGS], flags | (s_flags & 0xC0000000u));
    info[RK_INFO_SPLITS] = S;
    info[RK_INFO_LEAVES] = leaves;
    info[5] = nlev;
  }
}

__device__ __forceinline__ void store_rbox(float* __restrict__ p, const float (&mn)[3], const float (&mx)[3]) {
  float2* o = reinterpret_cast<float2*>(p);  // 24 B per record: 8-B aligned
  o[0] = make_float2(mn[0], mn[1]);
  o[1] = make_float2(mn[2], mx[0]);
  o[2] = make_float2(mx[1], mx[2]);
}

// Leaf boxes (kernel_calcBoundingBoxes pass 0, CUDA_buildMeshTreeLBVH.cu:246-268):
// merge of the leaf's triangle boxes via indices. One wave per record; leaves of
// more than kWaveLeaf faces, which only incomplete trees (the Hybrid's first
// pass) have, by the whole workgroup: of the 1M-face heightfield's at depth 12
// the largest took one wave 343 us, this takes 31.
constexpr uint32_t kLeafThreads = 1024, kWaveLeaf = 512;
__global__ __launch_bounds__(kLeafThreads) void k_leaf_boxes(TopoWs w, int large, const uint32_t* __restrict__ info,
                                                             const uint32_t* __restrict__ indices,
                                                             const Box* __restrict__ boxes) {
  constexpr uint32_t kWaves = kLeafThreads / 64;
  __shared__ __attribute__((aligned(8))) float s_box[kWaves][6];
  __shared__ uint32_t s_first[kWaves], s_cnt[kWaves];
  const uint32_t R = info[RK_INFO_NODE_COUNT];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // The leaf's faces t, t + threads, ... in that order, kLeafFetch at a time with
  // all their loads issued first: a face costs two dependent loads (its index,
  // then its box). In every lane, the wave's box.
  auto merge = [&](uint32_t first, uint32_t cnt, uint32_t t, uint32_t threads, float (&mn)[3], float (&mx)[3]) {
    for (int q = 0; q < 3; ++q) {
      mn[q] = RK_HUGE;
      mx[q] = -RK_HUGE;
    }
    constexpr uint32_t kLeafFetch = 8;
    for (uint32_t i0 = t; i0 < cnt; i0 += threads * kLeafFetch) {
      uint32_t ix[kLeafFetch];
#pragma unroll
      for (uint32_t k = 0; k < kLeafFetch; ++k) ix[k] = i0 + threads * k < cnt ? indices[first + i0 + threads * k] : 0u;
#pragma unroll
      for (uint32_t k = 0; k < kLeafFetch; ++k) {
        if (i0 + threads * k < cnt) {
          const Box b = rk::load_box(boxes + ix[k]);
          mn[0] = rk::fmn(mn[0], b.mn.x); mn[1] = rk::fmn(mn[1], b.mn.y); mn[2] = rk::fmn(mn[2], b.mn.z);
          mx[0] = rk::fmx(mx[0], b.mx.x); mx[1] = rk::fmx(mx[1], b.mx.y); mx[2] = rk::fmx(mx[2], b.mx.z);
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        mn[q] = rk::fmn(mn[q], __shfl_xor(mn[q], off, 64));
        mx[q] = rk::fmx(mx[q], __shfl_xor(mx[q], off, 64));
      }
    }
  };
  // neighbours in a level, which are alike in size, go to different workgroups
  for (uint32_t base = blockIdx.x; base < R; base += gridDim.x * kWaves) {
    const uint32_t r = base + wave * gridDim.x;
    float mn[3], mx[3];
    uint32_t first = 0, cnt = 0;
    const bool leaf = r < R && !(w.rmeta[r] & kInternal);
    if (leaf) {
      first = w.ra[r];
      cnt = (w.rb[r] & ~kMedian) - first;
      if (!large || cnt <= kWaveLeaf) {
        merge(first, cnt, lane, 64, mn, mx);
        if (lane == 0) store_rbox(w.rbox + 6 * (size_t)r, mn, mx);
        cnt = 0;
      }
    }
    if (!large) continue;
    if (lane == 0) {
      s_first[wave] = first;
      s_cnt[wave] = cnt;
    }
    __syncthreads();
    for (uint32_t x = 0; x < kWaves; ++x) {
      if (s_cnt[x] == 0u) continue;  // uniform
      merge(s_first[x], s_cnt[x], threadIdx.x, kLeafThreads, mn, mx);
      if (lane == 0) store_rbox(s_box[wave], mn, mx);
      __syncthreads();
      if (threadIdx.x == 0) {
        for (uint32_t v = 1; v < kWaves; ++v)
          for (int q = 0; q < 3; ++q) {
            mn[q] = rk::fmn(mn[q], s_box[v][q]);
            mx[q] = rk::fmx(mx[q], s_box[v][3 + q]);
          }
        store_rbox(w.rbox + 6 * (size_t)(base + x * gridDim.x), mn, mx);
      }
      __syncthreads();
    }
    __syncthreads();
  }
}

// Internal boxes, bottom-up by level in one workgroup. The fixpoint of the
// reference's real_depth racy passes (CUDA_buildMeshTreeLBVH.cu:269-301): a node
// takes the union of its children only if both have z-extent > 0, else it
// stays EMPTY (and so does every ancestor). Boxes are by record, so a level
// costs one dependent load (the children's two boxes, side by side), from LDS
// where the children's level fits, with the next level's kinds, children and leaf
// boxes loaded meanwhile. (By node id, three loads from memory per level: 50 us
// for the depth-12 tree of 1M faces; one: 33; 27 so.)
// Also counts the split bits before each kRankWords words, for k_emit_ref.
constexpr uint32_t kRefitPer = 3, kRefitLevel = kRefitPer * 1024;  // levels up to this size go through LDS
__global__ __launch_bounds__(1024) void k_refit_ref(TopoWs w, uint32_t n, const uint32_t* __restrict__ info) {
  __shared__ __attribute__((aligned(16))) float s_box[2][6 * kRefitLevel];
  __shared__ uint32_t s_tmp[16];
  __shared__ uint32_t s_lev[kMaxLevels + 2];
  const uint32_t nlev = info[5];
  uint32_t run = 0;
  const uint32_t groups = n / 32u / kRankWords + 1u;
  for (uint32_t g0 = 0; g0 < groups; g0 += 1024) {
    const uint32_t g = g0 + threadIdx.x;
    uint32_t c = 0;
    if (g < groups) {
      const uint4* p = reinterpret_cast<const uint4*>(w.bits + (size_t)g * kRankWords);
#pragma unroll
      for (uint32_t k = 0; k < kRankWords / 4; ++k) {
        const uint4 v = p[k];
        c += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
      }
    }
    uint32_t total;
    const uint32_t ex = block_excl_scan1024(c, s_tmp, &total);
    if (g < groups) w.ranks[g] = run + ex;
    run += total;
  }
  for (uint32_t k = threadIdx.x; k <= nlev; k += 1024) s_lev[k] = w.lev_begin[k];
  __syncthreads();
  uint32_t meta[kRefitPer], child[kRefitPer];
  float2 own[kRefitPer][3];
  // kinds, children and boxes (a leaf's; an internal node's is not there yet) of a level
  auto fetch = [&](int lv) {
    const uint32_t b0 = s_lev[lv], b1 = s_lev[lv + 1];
#pragma unroll
    for (uint32_t u = 0; u < kRefitPer; ++u) {
      const uint32_t r = b0 + u * 1024 + threadIdx.x;
      if (r < b1) {
        meta[u] = w.rmeta[r];
        child[u] = w.rchild[r];
        const float2* p = reinterpret_cast<const float2*>(w.rbox + 6 * (size_t)r);
#pragma unroll
        for (int q = 0; q < 3; ++q) own[u][q] = p[q];
      }
    }
  };
  auto merge = [](const float2* p, float (&mn)[3], float (&mx)[3]) {
    const float2 l0 = p[0], l1 = p[1], l2 = p[2], q0 = p[3], q1 = p[4], q2 = p[5];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      mn[q] = RK_HUGE;
      mx[q] = -RK_HUGE;
    }
    if (l2.y - l1.x > 0.0f && q2.y - q1.x > 0.0f) {
      mn[0] = rk::fmn(l0.x, q0.x); mn[1] = rk::fmn(l0.y, q0.y); mn[2] = rk::fmn(l1.x, q1.x);
      mx[0] = rk::fmx(l1.y, q1.y); mx[1] = rk::fmx(l2.x, q2.x); mx[2] = rk::fmx(l2.y, q2.y);
    }
  };
  bool fetched = false, below = false;  // below: the level below is in s_box
  for (int lv = (int)nlev - 1; lv >= 0; --lv) {
    const uint32_t b0 = s_lev[lv], b1 = s_lev[lv + 1];
    if (b1 - b0 <= kRefitLevel) {
      if (!fetched) fetch(lv);
      float* to = s_box[lv & 1];
      const float* from = s_box[(lv & 1) ^ 1];
#pragma unroll
      for (uint32_t u = 0; u < kRefitPer; ++u) {
        const uint32_t i = u * 1024 + threadIdx.x;
        if (b0 + i >= b1) continue;
        float mn[3], mx[3];
        if (meta[u] & kInternal) {
          merge(reinterpret_cast<const float2*>(below ? from + 6 * (child[u] - b1) : w.rbox + 6 * (size_t)child[u]),
                mn, mx);
          store_rbox(w.rbox + 6 * (size_t)(b0 + i), mn, mx);
        } else {
          mn[0] = own[u][0].x; mn[1] = own[u][0].y; mn[2] = own[u][1].x;
          mx[0] = own[u][1].y; mx[1] = own[u][2].x; mx[2] = own[u][2].y;
        }
        store_rbox(to + 6 * i, mn, mx);
      }
      fetched = lv > 0 && b0 - s_lev[lv - 1] <= kRefitLevel;
      if (fetched) fetch(lv - 1);
      below = true;
      if (fetched || lv == 0) lds_barrier();
      else __syncthreads();
    } else {
      for (uint32_t r = b0 + threadIdx.x; r < b1; r += 1024) {
        if (!(w.rmeta[r] & kInternal)) continue;
        float mn[3], mx[3];
        merge(reinterpret_cast<const float2*>(w.rbox + 6 * (size_t)w.rchild[r]), mn, mx);
        store_rbox(w.rbox + 6 * (size_t)r, mn, mx);
      }
      fetched = below = false;
      __syncthreads();
    }
  }
}

// The node records (make_node / make_leaf, :85-109), by the reference's ids:
// the internal node of preorder rank R gets children 2R+1, 2R+2 (:325-326,
// :394-395). R counts the internal nodes before it in preorder: those whose
// split is at or before its start a (in order, as many as leaves before a),
// and its ancestors it lies to the left of. So each record finds its own.
__global__ __launch_bounds__(256) void k_emit_ref(TopoWs w, const uint32_t* __restrict__ info,
                                                  Node* __restrict__ nodes) {
  __shared__ uint32_t s_lev[kMaxLevels + 2];
  const uint32_t R = info[RK_INFO_NODE_COUNT], nlev = info[5];
  for (uint32_t k = threadIdx.x; k <= nlev; k += 256) s_lev[k] = w.lev_begin[k];
  __syncthreads();
  auto rank_of = [&](uint32_t a, uint32_t meta) {
    const uint32_t word = a >> 5, g = word / kRankWords;
    uint32_t c = w.ranks[g] + (meta >> 1);
#pragma unroll
    for (uint32_t k = 0; k < kRankWords; ++k) {
      const uint32_t i = g * kRankWords + k;
      const uint32_t v = w.bits[i];
      c += __popc(i < word ? v : (i == word ? v & (0xFFFFFFFFu >> (31u - (a & 31u))) : 0u));
    }
    return c;
  };
  auto emit = [&](uint32_t r, uint32_t id, uint32_t level) {
    const uint32_t a = w.ra[r], meta = w.rmeta[r];
    Node nd;
    if (meta & kInternal) {
      nd.w0 = ((level % 3u) & 3u) << 1;
      nd.w1 = 2 * rank_of(a, meta) + 1;
    } else {
      nd.w0 = 1u | (((w.rb[r] & ~kMedian) - a) << 1);
      nd.w1 = a;
    }
    const float* b = w.rbox + 6 * (size_t)r;
    for (int q = 0; q < 3; ++q) {
      nd.bmin[q] = b[q];
      nd.bmax[q] = b[3 + q];
    }
    nodes[id] = nd;
  };
  for (uint32_t r = blockIdx.x * 256 + threadIdx.x; r < R; r += gridDim.x * 256) {
    if (r == 0) emit(0, 0, 0);
    const uint32_t meta = w.rmeta[r];
    if (!(meta & kInternal)) continue;
    uint32_t lo = 0, hi = nlev;  // the last level that starts at or before r
    while (lo + 1 < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_lev[mid] <= r) lo = mid;
      else hi = mid;
    }
    const uint32_t id = 2 * rank_of(w.ra[r], meta) + 1, c = w.rchild[r];
    emit(c, id, lo + 1);
    emit(c + 1, id + 1, lo + 1);
  }
}

__global__ __launch_bounds__(256) void k_gather_faces(const uint4* __restrict__ src, const uint32_t* __restrict__ idx,
                                                      uint4* __restrict__ dst, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}
__global__ __launch_bounds__(256) void k_copy_faces(const uint4* __restrict__ src, uint4* __restrict__ dst, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

inline unsigned blocks_for(uint32_t n, uint32_t per) { return (n + per - 1) / per; }

}  // namespace

extern "C" rk_status rk_calc_mesh_boxes(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                        uint32_t count, rk_aabox* boxes, uint32_t* indices) {
  if (count == 0) return RK_SUCCESS;
  if (!faces || !vertices || !boxes || !indices) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL(k_calc_boxes, dim3(blocks_for(count, 256)), dim3(256), 0, rk_hip_stream(stream),
                     reinterpret_cast<const uint4*>(faces), reinterpret_cast<const float4*>(vertices), count,
                     reinterpret_cast<Box*>(boxes), indices);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" rk_status rk_calc_morton_codes(rk_stream stream, const rk_aabox* boxes, uint32_t count,
                                          const rk_aabox* root_box, int mode, void* codes) {
  if (count == 0) return RK_SUCCESS;
  if (!boxes || !root_box || !codes || mode < 0 || mode > 2) return RK_ERROR_INVALID_VALUE;
  float4 rmin = make_float4(root_box->min.x, root_box->min.y, root_box->min.z, root_box->min.w);
  float4 rmax = make_float4(root_box->max.x, root_box->max.y, root_box->max.z, root_box->max.w);
  hipLaunchKernelGGL(k_morton, dim3(blocks_for(count, 256)), dim3(256), 0, rk_hip_stream(stream),
                     reinterpret_cast<const Box*>(boxes), count, rmin, rmax, mode, codes);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" size_t rk_reorder_workspace_size(uint32_t count) { return rk_align_up((size_t)(count ? count : 1) * 16) + 256; }

extern "C" rk_status rk_reorder_mesh_faces(rk_stream stream, rk_uint4* faces, const uint32_t* indices, uint32_t count,
                                           void* ws, size_t ws_bytes) {
  if (count == 0) return RK_SUCCESS;
  if (!faces || !indices) return RK_ERROR_INVALID_VALUE;
  RkArena ar(ws, ws_bytes);
  uint4* tmp = ar.take<uint4>(count);
  if (!tmp) return RK_ERROR_WORKSPACE;
  hipStream_t st = rk_hip_stream(stream);
  uint4* f = reinterpret_cast<uint4*>(faces);
  hipLaunchKernelGGL(k_gather_faces, dim3(blocks_for(count, 256)), dim3(256), 0, st, f, indices, tmp, count);
  RK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_copy_faces, dim3(blocks_for(count, 256)), dim3(256), 0, st, tmp, f, count);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" size_t rk_build_lbvh_workspace_size(uint32_t face_count) {
  size_t n = face_count ? face_count : 1;
  size_t cap = 2 * n;
  size_t b = 0;
  b += rk_align_up(n * 4);            // codes
  b += rk_align_up(n * 4) * 2;        // level keys, positions
  b += rk_align_up(64 * 4);           // level counts
  b += rk_align_up(cap * 4) * 7;      // topology records: 24-B boxes, range starts
  b += rk_align_up((kMaxLevels + 2) * 4);
  b += rk_align_up(n * 4);            // record kinds, split bits and their ranks
  b += rk_align_up(n * 16);           // face reorder temp
  b += rk_sort_workspace_size((uint32_t)n, 4);
  return b + 4096;
}

extern "C" rk_status rk_build_lbvh(rk_stream stream, rk_uint4* faces, const rk_float4* vertices, uint32_t face_count,
                                   const rk_aabox* hitbox, int tree_complete, uint32_t tree_depth, rk_aabox* boxes,
                                   uint32_t* indices, rk_bvnode* nodes, uint32_t nodes_capacity, uint32_t* info,
                                   void* ws, size_t ws_bytes) {
  const uint32_t n = face_count;
  if (n == 0 || !faces || !vertices || !hitbox || !boxes || !indices || !nodes || !info) return RK_ERROR_INVALID_VALUE;
  if (tree_depth > 31) return RK_ERROR_INVALID_VALUE;
  if (n >= (1u << 30)) return RK_ERROR_UNSUPPORTED;
  if ((size_t)nodes_capacity < 2 * (size_t)n - 1) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  const size_t cap = 2 * (size_t)n;
  RkArena ar(ws, ws_bytes);
  uint32_t* codes = ar.take<uint32_t>(n);
  uint32_t* lev = ar.take<uint32_t>(n);
  uint32_t* pos = ar.take<uint32_t>(n);
  uint32_t* level_count = ar.take<uint32_t>(64);
  TopoWs tw;
  const size_t rec_bytes = 7 * rk_align_up(cap * 4);
  char* rec = ar.take<char>(rec_bytes);
  tw.lev_begin = ar.take<uint32_t>(kMaxLevels + 2);
  char* marks = ar.take<char>((size_t)n * 4);
  tw.cap = (uint32_t)cap;
  uint4* ftmp = ar.take<uint4>(n);
  size_t sort_bytes = rk_sort_workspace_size(n, 4);
  void* sort_ws = ar.take<char>(sort_bytes);
  if (!codes || !lev || !pos || !level_count || !rec || !tw.lev_begin || !marks || !ftmp || !sort_ws)
    return RK_ERROR_WORKSPACE;
  // The records: boxes and range starts in rec, which the sort of the splits
  // by level has as its workspace before; ends and children in the code sort's
  // and in codes and lev, done with by then; one byte each, the split bits and
  // their ranks in marks.
  const uint32_t groups = n / 32u / kRankWords + 1u;
  tw.rbox = reinterpret_cast<float*>(rec);
  tw.ra = reinterpret_cast<uint32_t*>(rec + 6 * rk_align_up(cap * 4));
  tw.rb = reinterpret_cast<uint32_t*>(sort_ws);  // at least 8 bytes per face
  tw.rchild = codes;
  tw.rmeta = reinterpret_cast<uint8_t*>(marks);
  tw.bits = reinterpret_cast<uint32_t*>(marks + ((cap + 63) & ~(size_t)63));
  tw.ranks = tw.bits + (size_t)groups * kRankWords;  // ends within marks, a multiple of 256 B, for every n

  rk_status s;
  const float4 rmin = make_float4(hitbox->min.x, hitbox->min.y, hitbox->min.z, hitbox->min.w);
  const float4 rmax = make_float4(hitbox->max.x, hitbox->max.y, hitbox->max.z, hitbox->max.w);
  uint4* f = reinterpret_cast<uint4*>(faces);
  // CUDA_radixSortGeneral(codes, indices, N, 32, true), CUDA_buildMeshTreeLBVH.cu:522-528: above its bitonic
  // class (32768) a stable sort, whose digits the box kernel counts. The sort of the splits by level has its
  // workspace in the topology's records, which nothing uses before that.
  const bool plain = n > 4u * 8192u;
  RkSortPlan<uint32_t> codes_plan, levels_plan;
  if (plain && (s = rk_sort_plan<uint32_t>(n, 32, false, codes, indices, sort_ws, sort_bytes, codes_plan)) != RK_SUCCESS)
    return s;
  if (n > 1 && (s = rk_sort_plan<uint32_t>(n - 1, 8, true, lev, pos, rec, rec_bytes, levels_plan)) !=
                   RK_SUCCESS)
    return s;
  const bool counted = n > 1 && !levels_plan.one;  // the levels are counted where they are found
  const size_t clear_a = plain ? codes_plan.head_words + codes_plan.status_words : 0;
  const size_t clear_b = counted ? levels_plan.head_words + levels_plan.status_words : 0;
  hipLaunchKernelGGL(k_lbvh_clear, dim3(std::min<unsigned>(1024u, blocks_for((uint32_t)(clear_a + clear_b + 64), 1024))),
                     dim3(256), 0, st, info, level_count, codes_plan.head, clear_a, levels_plan.head, clear_b, tw.bits,
                     groups * kRankWords);
  RK_CHECK_LAUNCH();
  // 4 faces per thread from 2^18 on, where that still leaves a workgroup for most CUs
  const uint32_t per = n >= (1u << 18) ? 4u : 1u;
  hipLaunchKernelGGL(k_boxes_morton32, dim3(blocks_for(n, per * kBoxThreads)), dim3(kBoxThreads), 0, st, f,
                     reinterpret_cast<const float4*>(vertices), n, rmin, rmax, reinterpret_cast<Box*>(boxes), indices,
                     codes, per, plain ? codes_plan.head + 1 : (uint32_t*)nullptr, codes_plan.copies,
                     tree_complete ? ftmp : (uint4*)nullptr);
  RK_CHECK_LAUNCH();
  s = plain ? rk_sort_run<uint32_t>(st, codes_plan, true, info + RK_INFO_FLAGS)
            : rk_sort_general_impl(st, codes, indices, n, 32, 0, sort_ws, sort_bytes, info + RK_INFO_FLAGS);
  if (s != RK_SUCCESS) return s;
  if (n > 1) {
    hipLaunchKernelGGL(k_split_levels, dim3(blocks_for(n - 1, kSplitThreads * kSplitPer)), dim3(kSplitThreads), 0, st,
                       codes, n, levels_plan.src, levels_plan.vsrc, counted ? levels_plan.head + 1 : level_count,
                       counted ? levels_plan.copies : 1u);
    RK_CHECK_LAUNCH();
    s = rk_sort_run<uint32_t>(st, levels_plan, counted, info + RK_INFO_FLAGS);
    if (s != RK_SUCCESS) return s;
  }
  hipLaunchKernelGGL(k_topo_ref, dim3(1), dim3(kTopoThreads), 0, st, pos,
                     counted ? levels_plan.head + 1 : level_count, counted ? levels_plan.copies : 1u, n, tree_depth,
                     tree_complete, tw, info);
  RK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_leaf_boxes, dim3(std::min(512u, blocks_for(n, 1024))), dim3(kLeafThreads), 0, st, tw,
                     tree_complete ? 0 : 1, info, indices, reinterpret_cast<const Box*>(boxes));
  RK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_refit_ref, dim3(1), dim3(1024), 0, st, tw, n, info);
  RK_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_emit_ref, dim3(std::min(2048u, blocks_for(n, 8 * 256))), dim3(256), 0, st, tw, info,
                     reinterpret_cast<Node*>(nodes));
  RK_CHECK_LAUNCH();
  if (tree_complete) {  // CUDA_reorderMeshFaces, CUDA_buildMeshTreeLBVH.cu:669-676
    hipLaunchKernelGGL(k_gather_faces, dim3(blocks_for(n, 256)), dim3(256), 0, st, ftmp, indices, f, n);
    RK_CHECK_LAUNCH();
  }
  return RK_SUCCESS;
}
