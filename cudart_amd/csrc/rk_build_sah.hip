// Binned SAH build (CUDA_buildMeshTreeSAH, CUDA_buildMeshTreeSAH.cu:224-789)
// and the Hybrid refinement of LBVH leaves (kernel_initStack, :647-666), for
// gfx950. The reference processes one node per 32-thread block with thread 0
// doing the binning, sweep and partition serially, and a host round trip per
// level through a 4096-entry global stack. Here the tree is made first, without
// node ids, and numbered afterwards:
//   items of more than 1024 faces, level by level, cut into 1024-face chunks,
//   one workgroup per chunk:
//     k_sah_bins     32 bins per item: count + primitive-box bounds (LDS, then
//                    atomics); each face's bin and the chunk's counts are kept
//     k_sah_split    one half-wave per item, one lane per bin: the reference
//                    sweep (:424-474), leaf test (:479-496), children (:501-530)
//     k_sah_scatter  stable partition (bin <= m_min goes left, :572-594) into the
//                    other id buffer, and the children's centroid bounds
//   k_sah_subtrees   items of at most 1024 faces, start to end in one workgroup's
//                    LDS: every level below them
//   k_sah_number,    ids in breadth-first order and the node records, level by
//   k_sah_number_run level
// The 999,698-face heightfield takes 640 us: 12 levels of bins (11.5 us: the gather
// of the boxes, then LDS atomics), split (7: a chain of loads) and scatter (9.7: the
// same gather), subtrees 153 (instruction issue), numbering 70. With the items
// numbered as they were made (nine kernels per level, the boxes gathered in four
// of them, and again on each of 19 levels for the small items) it took 1750.
// Min/max are exact in any order, so the atomics and the sweep's scans
// reproduce the reference's serial merges; each cost is the reference's
// expression on the same values. Node numbering: a level's items are in queue
// order, and its k-th internal item takes children (count + 2k, count + 2k + 1),
// the breadth-first equivalent of the reference's atomicAdd(node_count, 2).
#include <algorithm>
#include <iterator>
#include <numeric>

#include "rk_device.h"

namespace {

using rk::Box;
using rk::Node;

constexpr uint32_t kChunk = 1024;
constexpr int kCT = 256;             // threads of the per-chunk kernels
constexpr int kPer = kChunk / kCT;   // faces per thread
constexpr int kBins = 32;
constexpr uint32_t kLeafMin = 16;    // MIN_LEAF_SIZE, :55
constexpr uint32_t kLeafMax = 224;   // MAX_LEAF_SIZE, :56
constexpr uint32_t kLevelMax = 4096; // deeper trees are refused

// An item's record. The split positions of the items are all different (the
// ranges are disjoint and both sides hold faces: the cost of a split with an
// empty side is not a number), so an item split at position p has its children
// in records 2p and 2p + 1, with nothing to allocate; the items that the build
// starts from come after them, at 2n.
struct Rec {
  float bmin[3], bmax[3];
  uint32_t lo, cnt;
};
static_assert(sizeof(Rec) == 32, "record is 32 B");
constexpr uint32_t kLeaf = 0xFFFFFFFFu;  // link of a leaf; else split | axis << 30

struct BigItem {  // of more than kChunk faces
  uint32_t rec, lo, hi, chunk_base;
  float bmin[3], bmax[3];
  uint32_t bref, pad;  // its centroid bounds
};
static_assert(sizeof(BigItem) == 48, "item is 48 B");
struct BigDec {
  int m_min;  // -1: leaf
  uint32_t lcount;
};

// Accumulators of the big items, kept empty between levels by who reads them
// last (k_sah_split): 32 bins of (count, 3 min, 3 max ordered ints) in kBinSlots
// copies, which an item's chunks update in turn so that fewer atomics meet on
// one address; centroid bounds (6 ordered ints) of both children, likewise.
constexpr int kBinSlots = 4;
constexpr int kBinWords = kBins * 7;
constexpr int kAccWords = kBinSlots * kBinWords;
constexpr int kBoundSlots = 8;
constexpr int kBoundWords = 6 * kBoundSlots;

constexpr int kCtlFlags = 0, kCtlDeep = 1, kCtlRoots = 2, kCtlLargest = 5, kCtlHist = 16;
// a tree of n faces has fewer than n levels with internal items
__device__ __host__ constexpr size_t ctl_words(uint32_t n) { return kCtlHist + (n < kLevelMax ? n : kLevelMax) + 1; }
// per level parity: big items, their chunks
__device__ __host__ constexpr int kCtlBig(uint32_t par) { return 8 + 2 * (int)par; }
constexpr int kCtlRead = 12;  // words the host reads between levels

// Items of at most kChunk faces by size, so that a workgroup of k_sah_subtrees
// takes 8, 4 or 1 of them.
constexpr uint32_t kClasses = 3;
__device__ __host__ constexpr uint32_t class_cap(uint32_t c) { return c == 0 ? 128u : (c == 1 ? 256u : kChunk); }
__device__ __forceinline__ uint32_t class_of(uint32_t size) { return size <= 128u ? 0u : (size <= 256u ? 1u : 2u); }

struct Sah {
  uint32_t n, chunks_cap, big_cap;
  size_t m_cap;
  const Box* boxes;
  uint32_t *ids0, *ids1;  // levels of even parity read the first and write the second
  Rec* rec;
  uint32_t* link;
  uint32_t* node0;        // node ids of the starting items
  uint32_t *q0, *q1;      // a level's splits, in order, by parity
  uint2* roots;           // kClasses lists of (record, level)
  BigItem *big0, *big1;
  BigDec* dec;
  uint32_t *chunk_item0, *chunk_item1;
  int* acc;
  int *bnd0, *bnd1;
  uint16_t* cum;          // [bin][chunk]: faces of the chunk up to the bin
  uint8_t* bin;           // by position
  uint32_t* ctl;          // ctl_words; at kCtlHist the internal items per level
  uint32_t* groups;       // 3 x group_cap: internal items per kNumberItems of a level
  uint32_t group_cap;
};
constexpr uint32_t kNumberItems = 1024;

__device__ __forceinline__ BigItem* big_of(const Sah& s, uint32_t par) { return par ? s.big1 : s.big0; }
__device__ __forceinline__ uint32_t* chunks_of(const Sah& s, uint32_t par) {
  return par ? s.chunk_item1 : s.chunk_item0;
}
__device__ __forceinline__ int* bounds_of(const Sah& s, uint32_t par) { return par ? s.bnd1 : s.bnd0; }
__device__ __forceinline__ uint32_t* ids_of(const Sah& s, uint32_t par) { return par ? s.ids1 : s.ids0; }

__device__ __forceinline__ int f2o(float f) {  // order-preserving float -> int
  int i = __float_as_int(f);
  return i >= 0 ? i : (i ^ 0x7FFFFFFF);
}
__device__ __forceinline__ float o2f(int i) { return __int_as_float(i >= 0 ? i : (i ^ 0x7FFFFFFF)); }

__device__ __forceinline__ float box_area(float mnx, float mny, float mnz, float mxx, float mxy, float mxz) {
  float vx = mxx - mnx, vy = mxy - mny, vz = mxz - mnz;  // CUDABox.h:35-44
  return 2.f * (vx * vy + vx * vz + vy * vz);
}

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_tmp, uint32_t* total, int nthreads) {
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(incl, off, 64);
    if (lane >= (uint32_t)off) incl += y;
  }
  if (lane == 63) s_tmp[wave] = incl;
  __syncthreads();
  uint32_t wprefix = 0, tot = 0;
  for (int w = 0; w < nthreads / 64; ++w) {
    uint32_t c = s_tmp[w];
    wprefix += ((uint32_t)w < wave) ? c : 0u;
    tot += c;
  }
  __syncthreads();
  *total = tot;
  return wprefix + incl - v;
}

// Empties the accumulators, clears the counters and info, and makes the root
// item (root: not Hybrid).
__global__ __launch_bounds__(256) void k_sah_clear(Sah s, uint32_t* __restrict__ info, int root, float4 rmin,
                                                   float4 rmax) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256;
  const int lo = f2o(RK_HUGE), hi = f2o(-RK_HUGE);
  for (size_t i = t; i < (size_t)s.big_cap * kAccWords; i += stride) {
    const uint32_t k = (uint32_t)(i % 7);
    s.acc[i] = k == 0 ? 0 : (k < 4 ? lo : hi);
  }
  for (size_t i = t; i < (size_t)s.big_cap * 2 * kBoundWords; i += stride)
    s.bnd0[i] = s.bnd1[i] = i % 6 < 3 ? lo : hi;
  const uint32_t nch = root && s.n > kChunk ? (s.n + kChunk - 1) / kChunk : 0u;
  for (size_t i = t; i < ctl_words(s.n); i += stride) {
    uint32_t v = 0;
    if (nch && i == (size_t)kCtlBig(0)) v = 1;
    if (nch && i == (size_t)kCtlBig(0) + 1) v = nch;
    if (root && !nch && i == kCtlRoots + class_of(s.n)) v = 1;
    s.ctl[i] = v;
  }
  if (t < RK_INFO_WORDS) info[t] = 0u;
  for (size_t i = t; i < nch; i += stride) s.chunk_item0[i] = 0u;
  if (root && t == 0) {
    Rec r;
    r.bmin[0] = rmin.x; r.bmin[1] = rmin.y; r.bmin[2] = rmin.z;
    r.bmax[0] = rmax.x; r.bmax[1] = rmax.y; r.bmax[2] = rmax.z;
    r.lo = 0;
    r.cnt = s.n;
    s.rec[2 * (size_t)s.n] = r;
    s.node0[0] = 0;
    if (nch) {
      BigItem b;
      b.rec = 2 * s.n; b.lo = 0; b.hi = s.n; b.chunk_base = 0; b.bref = 0; b.pad = 0;
      for (int q = 0; q < 3; ++q) { b.bmin[q] = r.bmin[q]; b.bmax[q] = r.bmax[q]; }
      s.big0[0] = b;
    } else {
      s.roots[class_of(s.n) * s.m_cap] = make_uint2(2 * s.n, 0u);
    }
  }
}

// Hybrid entry (kernel_initStack, :647-666): every leaf of the existing tree
// becomes an item, in ascending node order, with the leaf's box.
__global__ __launch_bounds__(1024) void k_sah_init_from_leaves(Sah s, const Node* __restrict__ nodes,
                                                               uint32_t existing) {
  __shared__ uint32_t s_tmp[16], s_cnt[2 + kClasses], s_largest;
  if (threadIdx.x < 2 + kClasses) s_cnt[threadIdx.x] = 0;
  if (threadIdx.x == 0) s_largest = 0;
  uint32_t carry = 0;
  __syncthreads();
  for (uint32_t c0 = 0; c0 < existing; c0 += 1024) {
    const uint32_t k = c0 + threadIdx.x, lane = threadIdx.x & 63;
    uint32_t leaf = 0;
    Node nd;
    if (k < existing) {
      nd = nodes[k];
      leaf = rk::node_is_leaf(nd.w0);
    }
    uint32_t total;
    const uint32_t i = carry + block_excl_scan(leaf, s_tmp, &total, 1024);
    carry += total;
    uint32_t nch = 0, base = 0, at = 0;
    if (leaf) {
      Rec r;
      for (int q = 0; q < 3; ++q) { r.bmin[q] = nd.bmin[q]; r.bmax[q] = nd.bmax[q]; }
      r.lo = nd.w1;
      r.cnt = rk::leaf_count(nd.w0);
      const uint32_t rec = 2 * s.n + i;
      s.rec[rec] = r;
      s.node0[i] = k;
      if (r.cnt > kChunk) {
        nch = (r.cnt + kChunk - 1) / kChunk;
        at = atomicAdd(&s_cnt[0], 1u);
        base = atomicAdd(&s_cnt[1], nch);
        atomicMax(&s_largest, r.cnt);
        BigItem b;
        b.rec = rec; b.lo = r.lo; b.hi = r.lo + r.cnt; b.chunk_base = base; b.bref = at; b.pad = 0;
        for (int q = 0; q < 3; ++q) { b.bmin[q] = r.bmin[q]; b.bmax[q] = r.bmax[q]; }
        s.big0[at] = b;
      } else {
        const uint32_t c = class_of(r.cnt);
        s.roots[c * s.m_cap + atomicAdd(&s_cnt[2 + c], 1u)] = make_uint2(rec, 0u);
      }
    }
    for (uint64_t m = __ballot(nch != 0u); m; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      const uint32_t b = __shfl(base, l, 64), e = __shfl(nch, l, 64), a = __shfl(at, l, 64);
      for (uint32_t j = lane; j < e; j += 64) s.chunk_item0[b + j] = a;
    }
  }
  __syncthreads();
  if (threadIdx.x < 2) s.ctl[kCtlBig(0) + threadIdx.x] = s_cnt[threadIdx.x];
  else if (threadIdx.x < 2 + kClasses) s.ctl[kCtlRoots + threadIdx.x - 2] = s_cnt[threadIdx.x];
  else if (threadIdx.x == 64) s.ctl[kCtlLargest] = s_largest;
}

struct ChunkRange { BigItem it; uint32_t item, j, lo, hi; bool ok; };

__device__ __forceinline__ ChunkRange chunk_range(const Sah& s, uint32_t par) {
  ChunkRange r;
  r.ok = blockIdx.x < s.ctl[kCtlBig(par) + 1];
  if (!r.ok) return r;
  r.item = chunks_of(s, par)[blockIdx.x];
  r.it = big_of(s, par)[r.item];
  r.j = blockIdx.x - r.it.chunk_base;
  r.lo = r.it.lo + r.j * kChunk;
  r.hi = min(r.it.hi, r.lo + kChunk);
  return r;
}

__device__ __forceinline__ float center_axis(const Box& b, int a) {  // 0.5f * (min + max), :292
  return a == 0 ? (b.mn.x + b.mx.x) * 0.5f : (a == 1 ? (b.mn.y + b.mx.y) * 0.5f : (b.mn.z + b.mx.z) * 0.5f);
}

// Axis and bin scale of an item from its centroid bounds (:302-342).
__device__ __forceinline__ void item_axis(const int (&a)[6], int& axis, float& scale, float& bmin0) {
  float ex = o2f(a[3]) - o2f(a[0]), ey = o2f(a[4]) - o2f(a[1]), ez = o2f(a[5]) - o2f(a[2]);
  if (ex > ey) axis = (ex > ez) ? 0 : 2;
  else axis = (ey > ez) ? 1 : 2;
  float e = axis == 0 ? ex : (axis == 1 ? ey : ez);
  scale = (float)(kBins - 1) / e;
  bmin0 = o2f(a[axis]);
}

__device__ __forceinline__ int bin_of(const Box& b, int axis, float scale, float bmin0) {  // :375-385
  // truncated and clamped to [0, kBins - 1], NaN to 0 (fmaxf takes the number)
  return (int)fminf(fmaxf((center_axis(b, axis) - bmin0) * scale, 0.f), (float)(kBins - 1));
}

// A workgroup's centroid bounds into one of an item's copies.
__device__ __forceinline__ void add_bounds(int (&b)[6], int* __restrict__ bounds) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      b[q] = min(b[q], __shfl_xor(b[q], off, 64));
      b[3 + q] = max(b[3 + q], __shfl_xor(b[3 + q], off, 64));
    }
  __shared__ int s_red[16][6];
  if ((threadIdx.x & 63) == 0)
    for (int q = 0; q < 6; ++q) s_red[threadIdx.x >> 6][q] = b[q];
  __syncthreads();
  if (threadIdx.x < 6) {
    const int q = (int)threadIdx.x;
    int v = s_red[0][q];
    for (uint32_t w = 1; w < blockDim.x / 64; ++w) v = q < 3 ? min(v, s_red[w][q]) : max(v, s_red[w][q]);
    int* g = bounds + 6 * (blockIdx.x % kBoundSlots) + q;
    if (q < 3) atomicMin(g, v);
    else atomicMax(g, v);
  }
}

// Centroid bounds of the starting items (Hybrid; the root's come from
// k_boxes_root); those of the others come from k_sah_scatter.
__global__ __launch_bounds__(kCT) void k_sah_bounds(Sah s) {
  const ChunkRange r = chunk_range(s, 0);
  if (!r.ok) return;
  int b[6] = {f2o(RK_HUGE), f2o(RK_HUGE), f2o(RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE)};
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t l = r.lo + threadIdx.x + (uint32_t)u * kCT;
    if (l >= r.hi) continue;
    const Box x = rk::load_box(s.boxes + s.ids0[l]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int c = f2o(center_axis(x, q));
      b[q] = min(b[q], c);
      b[3 + q] = max(b[3 + q], c);
    }
  }
  add_bounds(b, s.bnd1 + (size_t)r.it.bref * kBoundWords);
}

// An item's centroid bounds from their copies.
__device__ __forceinline__ void item_bounds(const int* __restrict__ a, int (&cb)[6]) {
  for (int q = 0; q < 6; ++q) cb[q] = a[q];
  for (int v = 1; v < kBoundSlots; ++v)
    for (int q = 0; q < 3; ++q) {
      cb[q] = min(cb[q], a[6 * v + q]);
      cb[3 + q] = max(cb[3 + q], a[6 * v + 3 + q]);
    }
}

// The boxes go into kBinCopies copies of the bins by lane: neighbours in space
// are neighbours in the list and fall into the same bin, and atomics on one
// address take turns.
constexpr int kBinCopies = 8, kBinStride = kBinWords + 8;
__global__ __launch_bounds__(kCT) void k_sah_bins(Sah s, uint32_t par) {
  __shared__ int s_bin[kBinCopies][kBinStride];
  __shared__ uint32_t s_sum[kBins];
  // the next level's counters, which k_sah_split adds to
  if (blockIdx.x == 0 && threadIdx.x < 2) s.ctl[kCtlBig(par ^ 1u) + threadIdx.x] = 0u;
  const ChunkRange r = chunk_range(s, par);
  if (!r.ok) return;
  uint32_t id[kPer];
  const uint32_t* ids = ids_of(s, par);
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t l = r.lo + threadIdx.x + (uint32_t)u * kCT;
    id[u] = l < r.hi ? ids[l] : 0u;
  }
  for (int w = threadIdx.x; w < kBinCopies * kBinStride; w += kCT) {
    const int k = (w % kBinStride) % 7;
    (&s_bin[0][0])[w] = k == 0 ? 0 : (k < 4 ? f2o(RK_HUGE) : f2o(-RK_HUGE));
  }
  Box bb[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if (r.lo + threadIdx.x + (uint32_t)u * kCT < r.hi) bb[u] = rk::load_box(s.boxes + id[u]);
  int cb[6];
  item_bounds(bounds_of(s, par ^ 1u) + (size_t)r.it.bref * kBoundWords, cb);
  int axis;
  float scale, bmin0;
  item_axis(cb, axis, scale, bmin0);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t l = r.lo + threadIdx.x + (uint32_t)u * kCT;
    if (l >= r.hi) continue;
    const Box& b = bb[u];
    const int m = bin_of(b, axis, scale, bmin0);
    s.bin[l] = (uint8_t)m;
    int* p = s_bin[threadIdx.x % kBinCopies] + m * 7;
    atomicAdd(p, 1);
    atomicMin(p + 1, f2o(b.mn.x)); atomicMin(p + 2, f2o(b.mn.y)); atomicMin(p + 3, f2o(b.mn.z));
    atomicMax(p + 4, f2o(b.mx.x)); atomicMax(p + 5, f2o(b.mx.y)); atomicMax(p + 6, f2o(b.mx.z));
  }
  __syncthreads();
  int* g = s.acc + (size_t)r.item * kAccWords + (blockIdx.x % kBinSlots) * kBinWords;
  for (int w = threadIdx.x; w < kBinWords; w += kCT) {
    const int k = w % 7;
    int v = s_bin[0][w];
#pragma unroll
    for (int c = 1; c < kBinCopies; ++c) {
      const int x = s_bin[c][w];
      v = k == 0 ? v + x : (k < 4 ? min(v, x) : max(v, x));
    }
    if (k == 0) {
      s_sum[w / 7] = (uint32_t)v;
      if (v) atomicAdd(g + w, v);
    } else if (k < 4) {
      if (v != f2o(RK_HUGE)) atomicMin(g + w, v);
    } else if (v != f2o(-RK_HUGE)) {
      atomicMax(g + w, v);
    }
  }
  __syncthreads();
  if (threadIdx.x < kBins) {
    uint32_t c = s_sum[threadIdx.x];
#pragma unroll
    for (int off = 1; off < kBins; off <<= 1) {
      const uint32_t y = __shfl_up(c, off, 32);
      if (threadIdx.x >= (uint32_t)off) c += y;
    }
    s.cum[(size_t)threadIdx.x * s.chunks_cap + blockIdx.x] = (uint16_t)c;
  }
}

// The reference's sweep over one item's bins (:424-474) and children boxes
// (:501-530), one lane per bin: lane k of each 32-lane half holds bin k
// (count, ordered-int box) of its half's item, and every lane of the half
// calls this. The left sweep's running box and count after bin k are the
// inclusive prefix at lane k, and the right sweep's after bin k the inclusive
// suffix; min, max and integer sums give the same values in any order, and
// each lane then evaluates the reference's area and cost expressions on those
// values. The reference keeps the first strict minimum of its sweep from bin
// 31 down, i.e. the largest split index among the minimal costs. The
// children's boxes are the prefix at the chosen split and the suffix after it.
struct Sweep {
  int m_min;  // -1: no finite cost below +huge
  float T_min;
  int lcount;
  float child[12];  // left min xyz, left max xyz, right min xyz, right max xyz
};

// A step of a prefix over 32 lanes: what the lanes' neighbours hold, 'old' where
// there is none. row_shr 1, 2, 4, 8 within 16 lanes, then row_bcast 15 across.
template <int kStep>
__device__ __forceinline__ int lane_step(int old, int x) {
  if constexpr (kStep < 4) return __builtin_amdgcn_update_dpp(old, x, 0x110 | 1 << kStep, 0xF, 0xF, false);
  else return __builtin_amdgcn_update_dpp(old, x, 0x142, 0xA, 0xF, false);
}
template <int kStep>
__device__ __forceinline__ float lane_step(float old, float x) {
  return __int_as_float(lane_step<kStep>(__float_as_int(old), __float_as_int(x)));
}
template <int kStep = 0>
__device__ __forceinline__ void prefix_box(int& n, float (&mn)[3], float (&mx)[3]) {
  n += lane_step<kStep>(0, n);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    mn[q] = rk::fmn(mn[q], lane_step<kStep>(mn[q], mn[q]));
    mx[q] = rk::fmx(mx[q], lane_step<kStep>(mx[q], mx[q]));
  }
  if constexpr (kStep < 4) prefix_box<kStep + 1>(n, mn, mx);
}
// The value of each half's last lane.
__device__ __forceinline__ int half_last(int x) {
  const int a = __builtin_amdgcn_readlane(x, 31), b = __builtin_amdgcn_readlane(x, 63);
  return (threadIdx.x & 32u) ? b : a;
}
// Smallest over each half-wave, in every lane.
template <int kStep = 0>
__device__ __forceinline__ int half_min(int x) {
  x = min(x, lane_step<kStep>(0x7FFFFFFF, x));
  if constexpr (kStep < 4) return half_min<kStep + 1>(x);
  else return half_last(x);
}

__device__ __forceinline__ Sweep sweep_bins(int cnt, const float (&bmn)[3], const float (&bmx)[3], float pa,
                                            uint32_t k) {
  // the right sweep runs over the bins in reverse: bin 31 - k in lane k
  const int rev = 31 - (int)k;
  int lc = cnt, rc = __shfl(cnt, rev, 32);
  float lmn[3], lmx[3], rmn[3], rmx[3];
  for (int q = 0; q < 3; ++q) {
    lmn[q] = bmn[q];
    lmx[q] = bmx[q];
    rmn[q] = __shfl(bmn[q], rev, 32);
    rmx[q] = __shfl(bmx[q], rev, 32);
  }
  prefix_box(lc, lmn, lmx);
  prefix_box(rc, rmn, rmx);
  // cost of the split after bin k (k <= 30): prefix at k, suffix at k + 1
  const float rarea = 0.f + box_area(rmn[0], rmn[1], rmn[2], rmx[0], rmx[1], rmx[2]);
  const int next = (30 - (int)k) & 31;
  const float rarea_next = __shfl(rarea, next, 32);
  const int rc_next = __shfl(rc, next, 32);
  const float larea = 0.f + box_area(lmn[0], lmn[1], lmn[2], lmx[0], lmx[1], lmx[2]);
  const int lcount = 0 + lc;
  const float T = 1.0f * 2.f + 0.125f * ((larea / pa) * (float)lcount + (rarea_next / pa) * (float)(0 + rc_next));
  const bool valid = k < 31 && T < RK_HUGE;  // NaN and +huge never win a strict <
  // the smallest as an ordered int, then the largest index among the lanes that hold it as a number
  const float bt = o2f(half_min(valid ? f2o(T) : 0x7FFFFFFF));
  const uint32_t best = (uint32_t)(__ballot(valid && T == bt) >> (threadIdx.x & 32u));
  const int bj = best ? 31 - (int)__clz((int)best) : -1;
  Sweep r;
  r.m_min = bj;
  r.T_min = bj >= 0 ? bt : RK_HUGE;
  const int src_l = bj >= 0 ? bj : 0, src_r = bj >= 0 ? 30 - bj : 0;
  for (int q = 0; q < 3; ++q) {
    r.child[q] = __shfl(lmn[q], src_l, 32);
    r.child[3 + q] = __shfl(lmx[q], src_l, 32);
    r.child[6 + q] = __shfl(rmn[q], src_r, 32);
    r.child[9 + q] = __shfl(rmx[q], src_r, 32);
  }
  r.lcount = __shfl(lc, src_l, 32);
  return r;
}

// The leaf test (:479-496) on a sweep's result: the bin of the split, or -1. An
// item with no finite cut that is too large for a leaf becomes one anyway and is
// flagged (by the lane that says so).
__device__ __forceinline__ int split_bin(const Sah& s, uint32_t size, const Sweep& sw, bool flags) {
  if (size < kLeafMax && sw.T_min > (float)(size + 1) * 0.125f) return -1;
  // a split with an empty side never has a finite cost; the build ends for this reason
  const bool cut = sw.m_min >= 0 && sw.lcount > 0 && (uint32_t)sw.lcount < size;
  if (!cut && flags) atomicOr(s.ctl + kCtlFlags, (uint32_t)RK_FLAG_SAH_NO_CUT);
  return cut ? sw.m_min : -1;
}

// The child of this lane (0: left, 1: right) of a half-wave's item.
__device__ __forceinline__ Rec child_rec(const Sweep& sw, uint32_t k, uint32_t lo, uint32_t size) {
  Rec r;
  for (int q = 0; q < 3; ++q) {
    r.bmin[q] = k == 0 ? sw.child[q] : sw.child[6 + q];
    r.bmax[q] = k == 0 ? sw.child[3 + q] : sw.child[9 + q];
  }
  r.lo = k == 0 ? lo : lo + (uint32_t)sw.lcount;
  r.cnt = k == 0 ? (uint32_t)sw.lcount : size - (uint32_t)sw.lcount;
  return r;
}

// The decision on the level's big items, their children, and the next level's
// big items and chunks, in any order: one half-wave per item.
constexpr uint32_t kSplitItems = 8;
__global__ __launch_bounds__(32 * kSplitItems) void k_sah_split(Sah s, uint32_t par, uint32_t level) {
  // children: of more than kChunk faces, their chunks, the others by class; internal items
  __shared__ uint32_t s_cnt[3 + kClasses], s_base[3 + kClasses];
  const uint32_t m = s.ctl[kCtlBig(par)];
  if (blockIdx.x * kSplitItems >= m) return;
  const uint32_t t = threadIdx.x, k = t & 31u, i = blockIdx.x * kSplitItems + (t >> 5);
  if (t < 3 + kClasses) s_cnt[t] = 0u;
  __syncthreads();
  const bool live = i < m;
  BigItem it;
  uint32_t size = 0;
  int axis = 0, cnt = 0;
  float pa = 0.f, bmn[3] = {RK_HUGE, RK_HUGE, RK_HUGE}, bmx[3] = {-RK_HUGE, -RK_HUGE, -RK_HUGE};
  if (live) {
    it = big_of(s, par)[i];
    size = it.hi - it.lo;
    int* g = bounds_of(s, par ^ 1u) + (size_t)it.bref * kBoundWords;
    int* a = s.acc + (size_t)i * kAccWords;
    int cb[6], bi[7];
    item_bounds(g, cb);
    float scale, bmin0;
    item_axis(cb, axis, scale, bmin0);
    for (int q = 0; q < 7; ++q) bi[q] = a[k * 7 + q];
    for (int v = 1; v < kBinSlots; ++v) {
      const int* b = a + v * kBinWords + k * 7;
      bi[0] += b[0];
      for (int q = 1; q < 4; ++q) bi[q] = min(bi[q], b[q]);
      for (int q = 4; q < 7; ++q) bi[q] = max(bi[q], b[q]);
    }
    cnt = bi[0];
    for (int q = 0; q < 3; ++q) { bmn[q] = o2f(bi[1 + q]); bmx[q] = o2f(bi[4 + q]); }
    pa = box_area(it.bmin[0], it.bmin[1], it.bmin[2], it.bmax[0], it.bmax[1], it.bmax[2]);
    // empty again for the levels after this one
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int w = (int)k; w < kAccWords; w += 32) a[w] = w % 7 == 0 ? 0 : (w % 7 < 4 ? f2o(RK_HUGE) : f2o(-RK_HUGE));
    for (int w = (int)k; w < kBoundWords; w += 32) g[w] = w % 6 < 3 ? f2o(RK_HUGE) : f2o(-RK_HUGE);
  }
  const Sweep sw = sweep_bins(cnt, bmn, bmx, pa, k);
  int m_min = -1;
  Rec child;
  uint32_t cls = 0, at = 0, nch = 0, chunk_at = 0;
  if (live) {
    m_min = split_bin(s, size, sw, k == 0);
    if (m_min >= 0 && k < 2) {
      child = child_rec(sw, k, it.lo, size);
      if (child.cnt > kChunk) {
        nch = (child.cnt + kChunk - 1) / kChunk;
        at = atomicAdd(&s_cnt[0], 1u);
        chunk_at = atomicAdd(&s_cnt[1], nch);
      } else {
        cls = class_of(child.cnt);
        at = atomicAdd(&s_cnt[3 + cls], 1u);
      }
      if (k == 0) {
        atomicAdd(&s_cnt[2], 1u);
        if (level >= kLevelMax) s.ctl[kCtlDeep] = 1u;
      }
    }
  }
  __syncthreads();
  if (t < 3 + kClasses && s_cnt[t]) {
    const uint32_t to = t < 2 ? kCtlBig(par ^ 1u) + t : (t == 2 ? kCtlHist + level : kCtlRoots + t - 3);
    s_base[t] = atomicAdd(s.ctl + to, s_cnt[t]);
  }
  __syncthreads();
  if (!live) return;
  if (k == 0) {
    BigDec d;
    d.m_min = m_min;
    d.lcount = (uint32_t)sw.lcount;
    s.dec[i] = d;
    s.link[it.rec] = m_min >= 0 ? (it.lo + (uint32_t)sw.lcount) | (uint32_t)axis << 30 : kLeaf;
  }
  if (m_min < 0) return;
  if (k < 2) {
    const uint32_t rec = 2 * (it.lo + (uint32_t)sw.lcount) + k;
    s.rec[rec] = child;
    if (nch) {
      at += s_base[0];
      chunk_at += s_base[1];
      BigItem b;
      b.rec = rec; b.lo = child.lo; b.hi = child.lo + child.cnt; b.chunk_base = chunk_at;
      b.bref = 2 * i + k;
      b.pad = 0;
      for (int q = 0; q < 3; ++q) { b.bmin[q] = child.bmin[q]; b.bmax[q] = child.bmax[q]; }
      big_of(s, par ^ 1u)[at] = b;
    } else {
      s.roots[cls * s.m_cap + s_base[3 + cls] + at] = make_uint2(rec, level + 1);
    }
  }
  uint32_t* map = chunks_of(s, par ^ 1u);
  for (int c = 0; c < 2; ++c) {
    const uint32_t b = __shfl(chunk_at, c, 32), e = __shfl(nch, c, 32), a = __shfl(at, c, 32);
    for (uint32_t j = k; j < e; j += 32) map[b + j] = a;
  }
}

// Smallest of each of 12 values over a wave, in a way that halves the values
// while it can: lane 0 ends with v[0..2], lane 16 with v[3..5], 32 with v[6..8],
// 48 with v[9..11], in v[0..2].
__device__ __forceinline__ void wave_min12(int (&v)[12], uint32_t lane) {
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const int send = lane & 32u ? v[q] : v[6 + q], keep = lane & 32u ? v[6 + q] : v[q];
    v[q] = min(keep, __shfl_xor(send, 32, 64));
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int send = lane & 16u ? v[q] : v[3 + q], keep = lane & 16u ? v[3 + q] : v[q];
    v[q] = min(keep, __shfl_xor(send, 16, 64));
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1)
#pragma unroll
    for (int q = 0; q < 3; ++q) v[q] = min(v[q], __shfl_xor(v[q], off, 64));
}

// The stable partition: a face's place needs the left faces of the item's
// earlier chunks (their cumulative bin counts at the split, one run of memory)
// and those before it in the chunk (ballots). A leaf's ids go to where the
// finished ones are.
__global__ __launch_bounds__(kCT) void k_sah_scatter(Sah s, uint32_t par) {
  constexpr uint32_t kWaves = kCT / 64;
  __shared__ uint32_t s_left[kWaves], s_before[kWaves];
  __shared__ int s_red[kWaves][4][3];
  const ChunkRange r = chunk_range(s, par);
  if (!r.ok) return;
  const BigDec d = s.dec[r.item];
  const uint32_t* src = ids_of(s, par);
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  if (d.m_min < 0) {
    if (par)
      for (uint32_t l = r.lo + t; l < r.hi; l += kCT) s.ids0[l] = src[l];
    return;
  }
  uint32_t id[kPer];
  int bin[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t l = r.lo + w * (64u * kPer) + (uint32_t)u * 64u + lane;
    id[u] = l < r.hi ? src[l] : 0u;
    bin[u] = l < r.hi ? (int)s.bin[l] : kBins;
  }
  const bool need_l = d.lcount > kChunk, need_r = r.it.hi - r.it.lo - d.lcount > kChunk;
  Box bb[kPer];
  if (need_l || need_r) {
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      if (bin[u] < kBins) bb[u] = rk::load_box(s.boxes + id[u]);
  }
  uint32_t before = 0;
  const uint16_t* cum = s.cum + (size_t)d.m_min * s.chunks_cap + r.it.chunk_base;
  for (uint32_t j = t; j < r.j; j += kCT) before += cum[j];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  uint64_t left[kPer];
  uint32_t mine = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    left[u] = __ballot(bin[u] <= d.m_min);
    mine += (uint32_t)__popcll(left[u]);
  }
  if (lane == 0) {
    s_left[w] = mine;
    s_before[w] = before;
  }
  if (need_l || need_r) {
    int v[12];  // left min, left max, right min, right max; ~x turns a max into a min
#pragma unroll
    for (int q = 0; q < 12; ++q) v[q] = q % 6 < 3 ? f2o(RK_HUGE) : ~f2o(-RK_HUGE);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      if (bin[u] >= kBins) continue;
      const bool is_left = bin[u] <= d.m_min;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int c = f2o(center_axis(bb[u], q)), lo = min(is_left ? v[q] : v[6 + q], c),
                  hi = min(is_left ? v[3 + q] : v[9 + q], ~c);
        v[q] = is_left ? lo : v[q];
        v[3 + q] = is_left ? hi : v[3 + q];
        v[6 + q] = is_left ? v[6 + q] : lo;
        v[9 + q] = is_left ? v[9 + q] : hi;
      }
    }
    wave_min12(v, lane);
    if ((lane & 15u) == 0)
      for (int q = 0; q < 3; ++q) s_red[w][lane >> 4][q] = v[q];
  }
  __syncthreads();
  if ((need_l || need_r) && t < 12) {
    const uint32_t part = t / 3, q = t % 3;
    int v = s_red[0][part][q];
    for (uint32_t x = 1; x < kWaves; ++x) v = min(v, s_red[x][part][q]);
    int* g = bounds_of(s, par) + (size_t)(2 * r.item + part / 2) * kBoundWords + 6 * (blockIdx.x % kBoundSlots) +
             3 * (part & 1u) + q;
    if (part < 2 ? need_l : need_r) {
      if (part & 1u) atomicMax(g, ~v);
      else atomicMin(g, v);
    }
  }
  uint32_t rank = 0;
  for (uint32_t x = 0; x < kWaves; ++x) rank += s_before[x] + (x < w ? s_left[x] : 0u);
  uint32_t* dst = ids_of(s, par ^ 1u);
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t l = r.lo + w * (64u * kPer) + (uint32_t)u * 64u + lane;
    const uint32_t lrank = rank + __builtin_amdgcn_mbcnt_hi((uint32_t)(left[u] >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)left[u], 0u));
    if (l < r.hi) dst[bin[u] <= d.m_min ? r.it.lo + lrank : r.it.lo + d.lcount + (l - r.it.lo - lrank)] = id[u];
    rank += (uint32_t)__popcll(left[u]);
  }
}

// Items of at most kChunk faces, to the leaves: a workgroup takes 1 of more than
// 256 faces, or 4 or 8 smaller ones, reads their boxes once into LDS and makes
// every level below them there. Items of more than kWide faces are done by the
// whole workgroup, then the others by half-waves (the sweep is a lane per bin),
// a round per level. A face is its place in the workgroup's lists at the start;
// s_ord holds the faces in order (by the item's depth below its root, odd and
// even), with the bin above.
// What bounds it is instruction issue: the sweep goes over lane rows (DPP), not
// through LDS (213 us, now 153 for the 1M-face heightfield); kWide 256, 512 and
// 1024: 157, 153, 162.
constexpr uint32_t kTreeThreads = 256, kTreeHalves = kTreeThreads / 32, kWide = 512;
constexpr uint32_t kTreeList = kChunk / (kLeafMin + 1) + 1;  // items that are not leaves by size
struct TreeItem {
  uint32_t range;  // lo | (size - 1) << 10
  uint32_t rec;
  float area;
  uint32_t depth;
};
struct RootsDone { uint32_t n[kClasses]; };  // of each list, taken by an earlier launch
__global__ __launch_bounds__(kTreeThreads, 4) void k_sah_subtrees(Sah s, RootsDone done) {
  __shared__ float s_box[6][kChunk];
  __shared__ uint16_t s_ord[2][kChunk];
  __shared__ int s_bins[kTreeHalves][kBinWords];
  __shared__ TreeItem s_list[2][kTreeList];
  __shared__ TreeItem s_wide[4];
  __shared__ uint32_t s_n[2], s_nwide;
  __shared__ uint32_t s_shift[8];   // global position less place, per 128 places
  __shared__ uint32_t s_size[8], s_rec[8], s_level[8];
  __shared__ uint32_t s_hist[8][32];  // internal items by depth below their root
  __shared__ uint32_t s_left[kTreeThreads / 64];
  __shared__ int s_red[kTreeHalves][6];
  __shared__ int s_cut, s_lcount;
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6, h = t >> 5, k = t & 31u;
  const uint32_t n0 = s.ctl[kCtlRoots] - done.n[0], n1 = s.ctl[kCtlRoots + 1] - done.n[1],
                 n2 = s.ctl[kCtlRoots + 2] - done.n[2];
  const uint32_t g0 = (n0 + 7) / 8, g1 = (n1 + 3) / 4;
  // the larger ones first
  for (uint32_t group = blockIdx.x; group < n2 + g1 + g0; group += gridDim.x) {
    const uint32_t cls = group < n2 ? 2u : (group < n2 + g1 ? 1u : 0u);
    const uint32_t cap = class_cap(cls), per = kChunk / cap;
    const uint32_t first = (group - (cls == 2 ? 0u : (cls == 1 ? n2 : n2 + g1))) * per;
    const uint32_t have = cls == 0 ? n0 - first : (cls == 1 ? n1 - first : 1u);  // may be more than per
    if (t < 8) s_size[t] = 0u;
    if (t < 2) s_n[t] = 0u;
    if (t == 2) s_nwide = 0u;
    (&s_hist[0][0])[t] = 0u;
    __syncthreads();
    if (t < per && t < have) {
      const uint2 root = s.roots[cls * s.m_cap + done.n[cls] + first + t];
      const Rec r = s.rec[root.x];
      s_size[t] = r.cnt;
      s_rec[t] = root.x;
      s_level[t] = root.y;
      for (uint32_t x = 0; x < cap / 128u; ++x) s_shift[t * (cap / 128u) + x] = r.lo - t * cap;
      if (r.cnt > kLeafMin) {
        TreeItem it;
        it.range = (t * cap) | (r.cnt - 1u) << 10;
        it.rec = root.x;
        it.area = box_area(r.bmin[0], r.bmin[1], r.bmin[2], r.bmax[0], r.bmax[1], r.bmax[2]);
        it.depth = 0;
        if (r.cnt > kWide) s_wide[atomicAdd(&s_nwide, 1u)] = it;
        else s_list[0][atomicAdd(&s_n[0], 1u)] = it;
      } else {
        s.link[root.x] = kLeaf;
      }
    }
    __syncthreads();
    {
      uint32_t id[kChunk / kTreeThreads];
      bool in[kChunk / kTreeThreads];
#pragma unroll
      for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
        const uint32_t l = t + u * kTreeThreads, x = l / cap;
        in[u] = l - x * cap < s_size[x];
        id[u] = 0;
        if (!in[u]) continue;
        // all ids end in ids0; ids1 keeps them until then
        const uint32_t g = s_shift[l >> 7] + l;
        if (s_level[x] & 1u) {
          id[u] = s.ids1[g];
          if (s_size[x] <= kLeafMin) s.ids0[g] = id[u];
        } else {
          id[u] = s.ids0[g];
          s.ids1[g] = id[u];
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
        const uint32_t l = t + u * kTreeThreads;
        if (!in[u]) continue;
        const Box b = rk::load_box(s.boxes + id[u]);
        s_box[0][l] = b.mn.x; s_box[1][l] = b.mn.y; s_box[2][l] = b.mn.z;
        s_box[3][l] = b.mx.x; s_box[4][l] = b.mx.y; s_box[5][l] = b.mx.z;
        s_ord[0][l] = (uint16_t)l;
      }
    }
    __syncthreads();

    // what goes between a wave's lanes through LDS
    auto wave_order = [] {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    auto load = [&](uint32_t f) {
      Box b;
      b.mn = make_float4(s_box[0][f], s_box[1][f], s_box[2][f], 0.f);
      b.mx = make_float4(s_box[3][f], s_box[4][f], s_box[5][f], 0.f);
      return b;
    };
    auto finish = [&](uint32_t place, uint32_t f) {
      s.ids0[s_shift[place >> 7] + place] = s.ids1[s_shift[f >> 7] + f];
    };
    auto add_bounds = [&](const Box& b, int (&c)[6]) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int x = f2o(center_axis(b, q));
        c[q] = min(c[q], x);
        c[3 + q] = max(c[3 + q], x);
      }
    };
    auto half_bounds = [](int (&c)[6]) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        c[q] = half_min(c[q]);
        c[3 + q] = ~half_min(~c[3 + q]);
      }
    };
    auto add_bin = [&](int* bins, const Box& b, int m) {
      int* p = bins + m * 7;
      atomicAdd(p, 1);
      atomicMin(p + 1, f2o(b.mn.x)); atomicMin(p + 2, f2o(b.mn.y)); atomicMin(p + 3, f2o(b.mn.z));
      atomicMax(p + 4, f2o(b.mx.x)); atomicMax(p + 5, f2o(b.mx.y)); atomicMax(p + 6, f2o(b.mx.z));
    };
    auto empty_bin = [](int q) { return q % 7 == 0 ? 0 : (q % 7 < 4 ? f2o(RK_HUGE) : f2o(-RK_HUGE)); };
    // by lanes 0 and 1 of a half-wave: the records and the items of the children
    auto children = [&](const TreeItem& it, const Sweep& sw, int axis, uint32_t lo, uint32_t size, bool wide,
                        uint32_t next) {
      const uint32_t x = lo / cap, gl = s_shift[lo >> 7] + lo, split = gl + (uint32_t)sw.lcount;
      const Rec r = child_rec(sw, k, gl, size);
      s.rec[2 * (size_t)split + k] = r;
      if (r.cnt <= kLeafMin) {
        s.link[2 * (size_t)split + k] = kLeaf;
      } else {
        TreeItem c;
        c.range = (k == 0 ? lo : lo + (uint32_t)sw.lcount) | (r.cnt - 1u) << 10;
        c.rec = 2 * split + k;
        c.area = box_area(r.bmin[0], r.bmin[1], r.bmin[2], r.bmax[0], r.bmax[1], r.bmax[2]);
        c.depth = it.depth + 1u;
        if (wide && r.cnt > kWide) s_wide[atomicAdd(&s_nwide, 1u)] = c;
        else s_list[next][atomicAdd(&s_n[next], 1u)] = c;
      }
      if (k == 0) {
        s.link[it.rec] = split | (uint32_t)axis << 30;
        const uint32_t level = s_level[x] + it.depth;
        if (it.depth < 32u) atomicAdd(&s_hist[x][it.depth], 1u);
        else if (level <= kLevelMax) atomicAdd(s.ctl + kCtlHist + level, 1u);
        if (level >= kLevelMax) s.ctl[kCtlDeep] = 1u;
      }
    };

    while (s_nwide != 0u) {
      const TreeItem it = s_wide[s_nwide - 1u];
      const uint32_t lo = it.range & 1023u, size = (it.range >> 10) + 1u, now = it.depth & 1u;
      int c[6] = {f2o(RK_HUGE), f2o(RK_HUGE), f2o(RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE)};
      uint32_t f[kChunk / kTreeThreads];
#pragma unroll
      for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
        const uint32_t l = w * 256u + u * 64u + lane;
        f[u] = l < size ? s_ord[now][lo + l] & 1023u : 0u;
      }
#pragma unroll
      for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
        if (w * 256u + u * 64u + lane >= size) continue;
        add_bounds(load(f[u]), c);
      }
      half_bounds(c);
      if (k == 0)
        for (int q = 0; q < 6; ++q) s_red[h][q] = c[q];
      for (int x = (int)k; x < kBinWords; x += 32) s_bins[h][x] = empty_bin(x);
      __syncthreads();
      if (t == 0) s_nwide -= 1u;
      for (int q = 0; q < 3; ++q)
        for (uint32_t x = 0; x < kTreeHalves; ++x) {
          c[q] = min(c[q], s_red[x][q]);
          c[3 + q] = max(c[3 + q], s_red[x][3 + q]);
        }
      int axis;
      float scale, bmin0;
      item_axis(c, axis, scale, bmin0);
      int bin[kChunk / kTreeThreads];
#pragma unroll
      for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
        bin[u] = kBins;
        if (w * 256u + u * 64u + lane >= size) continue;
        const Box b = load(f[u]);
        bin[u] = bin_of(b, axis, scale, bmin0);
        add_bin(s_bins[h], b, bin[u]);
      }
      __syncthreads();
      if (t < (uint32_t)kBinWords) {
        const int q = (int)t % 7;
        int v = s_bins[0][t];
        for (uint32_t x = 1; x < kTreeHalves; ++x) {
          const int y = s_bins[x][t];
          v = q == 0 ? v + y : (q < 4 ? min(v, y) : max(v, y));
        }
        s_bins[0][t] = v;
      }
      __syncthreads();
      Sweep sw;
      if (t < 64) {  // one wave: issue slots are what the kernel runs out of
        float bmn[3], bmx[3];
        const int* row = s_bins[0] + k * 7;
        for (int q = 0; q < 3; ++q) { bmn[q] = o2f(row[1 + q]); bmx[q] = o2f(row[4 + q]); }
        sw = sweep_bins(row[0], bmn, bmx, it.area, k);
        const int m = split_bin(s, size, sw, t == 0);
        if (t == 0) {
          s_cut = m;
          s_lcount = sw.lcount;
        }
      }
      __syncthreads();
      const int m_min = s_cut;
      if (m_min < 0) {
        if (t == 0) s.link[it.rec] = kLeaf;
        for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
          const uint32_t l = w * 256u + u * 64u + lane;
          if (l < size) finish(lo + l, f[u]);
        }
      } else {
        uint64_t left[kChunk / kTreeThreads];
        uint32_t mine = 0, rank = 0;
#pragma unroll
        for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
          left[u] = __ballot(bin[u] <= m_min);
          mine += (uint32_t)__popcll(left[u]);
        }
        if (lane == 0) s_left[w] = mine;
        __syncthreads();
        for (uint32_t x = 0; x < w; ++x) rank += s_left[x];
        const uint32_t lc = (uint32_t)s_lcount;
#pragma unroll
        for (uint32_t u = 0; u < kChunk / kTreeThreads; ++u) {
          const uint32_t l = w * 256u + u * 64u + lane;
          const uint32_t lrank = rank + __builtin_amdgcn_mbcnt_hi((uint32_t)(left[u] >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)left[u], 0u));
          const bool is_left = bin[u] <= m_min;
          const uint32_t place = lo + (is_left ? lrank : lc + (l - lrank));
          if (l < size) {
            s_ord[now ^ 1u][place] = (uint16_t)f[u];
            if ((is_left ? lc : size - lc) <= kLeafMin) finish(place, f[u]);
          }
          rank += (uint32_t)__popcll(left[u]);
        }
        if (t < 2) children(it, sw, axis, lo, size, true, 0);
      }
      __syncthreads();
    }

    uint32_t cur = 0, count = s_n[0];
    while (count != 0u) {
      for (uint32_t i = h; i < count; i += kTreeHalves) {
        const TreeItem it = s_list[cur][i];
        const uint32_t lo = it.range & 1023u, size = (it.range >> 10) + 1u, now = it.depth & 1u;
        uint16_t* ord = s_ord[now] + lo;
        int* bins = s_bins[h];
        int c[6] = {f2o(RK_HUGE), f2o(RK_HUGE), f2o(RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE)};
        for (uint32_t l = k; l < size; l += 32) add_bounds(load(ord[l] & 1023u), c);
        half_bounds(c);
        int axis;
        float scale, bmin0;
        item_axis(c, axis, scale, bmin0);
        for (int x = (int)k; x < kBinWords; x += 32) bins[x] = empty_bin(x);
        wave_order();
        for (uint32_t l = k; l < size; l += 32) {
          const uint32_t f = ord[l] & 1023u;
          const Box b = load(f);
          const int m = bin_of(b, axis, scale, bmin0);
          ord[l] = (uint16_t)(f | (uint32_t)m << 10);
          add_bin(bins, b, m);
        }
        wave_order();
        float bmn[3], bmx[3];
        const int* row = bins + k * 7;
        for (int q = 0; q < 3; ++q) { bmn[q] = o2f(row[1 + q]); bmx[q] = o2f(row[4 + q]); }
        const Sweep sw = sweep_bins(row[0], bmn, bmx, it.area, k);
        const int m_min = split_bin(s, size, sw, k == 0);
        if (m_min < 0) {
          if (k == 0) s.link[it.rec] = kLeaf;
          for (uint32_t l = k; l < size; l += 32) finish(lo + l, ord[l] & 1023u);
        } else {
          const uint32_t lc = (uint32_t)sw.lcount;
          uint32_t rank = 0;
          for (uint32_t l0 = 0; l0 < size; l0 += 32) {
            const uint32_t l = l0 + k, v = l < size ? ord[l] : 0xFFFFu;
            const bool is_left = (int)(v >> 10) <= m_min;
            const uint32_t left = (uint32_t)(__ballot(is_left) >> (lane & 32u));
            const uint32_t lrank = rank + (uint32_t)__popc(left & ((1u << k) - 1u));
            const uint32_t place = lo + (is_left ? lrank : lc + (l - lrank));
            if (l < size) {
              s_ord[now ^ 1u][place] = (uint16_t)(v & 1023u);
              if ((is_left ? lc : size - lc) <= kLeafMin) finish(place, v & 1023u);
            }
            rank += (uint32_t)__popc(left);
          }
          if (k < 2) children(it, sw, axis, lo, size, false, cur ^ 1u);
        }
        wave_order();
      }
      __syncthreads();
      count = s_n[cur ^ 1u];
      if (t == 0) s_n[cur] = 0u;
      cur ^= 1u;
      __syncthreads();
    }
    const uint32_t level = s_level[h] + k, c = s_hist[h][k];
    if (c && level <= kLevelMax) atomicAdd(s.ctl + kCtlHist + level, c);
    __syncthreads();
  }
}

// A level's items i of m (this thread's, in order): the node record, its id id0 + i
// (the starting items': node0), and the internal ones' splits in order to
// q[2 * rank]. before: internal items of the level before the workgroup's.
// Counts the next level's internal items by group, if there is a groups. Returns
// the workgroup's internal items.
__device__ __forceinline__ uint32_t number_items(const Sah& s, uint32_t level, uint32_t i, uint32_t m,
                                                 const uint32_t* q_in, uint32_t* q_out, uint32_t id0, uint32_t before,
                                                 uint32_t child0, uint32_t* groups, Node* __restrict__ nodes,
                                                 uint32_t nodes_cap, uint32_t* s_wave) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const bool in = i < m;
  Rec r;
  uint32_t link = kLeaf, id = 0;
  if (in) {
    const uint32_t rec = level ? 2 * q_in[i >> 1] + (i & 1u) : 2 * s.n + i;
    link = s.link[rec];
    r = s.rec[rec];
    id = level ? id0 + i : s.node0[i];
  }
  const bool internal = link != kLeaf;
  const uint64_t mask = __ballot(internal);
  if (lane == 0) s_wave[w] = (uint32_t)__popcll(mask);
  __syncthreads();
  uint32_t k =
      before + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
  uint32_t total = 0;
#pragma unroll
  for (uint32_t x = 0; x < 16; ++x) {
    const uint32_t c = s_wave[x];
    k += x < w ? c : 0u;
    total += c;
  }
  if (in) {
    Node nd;
    for (int q = 0; q < 3; ++q) { nd.bmin[q] = r.bmin[q]; nd.bmax[q] = r.bmax[q]; }
    nd.w0 = internal ? (link >> 30) << 1 : 1u | (r.cnt << 1);
    nd.w1 = internal ? child0 + 2 * k : r.lo;
    if (id < nodes_cap) nodes[id] = nd;
  }
  const uint32_t split = link & 0x3FFFFFFFu;
  if (internal) q_out[k] = split;
  if (groups && mask) {
    uint2 below = make_uint2(kLeaf, kLeaf);
    if (internal) below = *reinterpret_cast<const uint2*>(s.link + 2 * (size_t)split);
    const uint32_t g = 2 * k / kNumberItems, c = (below.x != kLeaf ? 1u : 0u) + (below.y != kLeaf ? 1u : 0u);
    const uint32_t g0 = (uint32_t)__shfl((int)g, __builtin_ctzll(mask), 64);  // a wave's children lie in two groups
    const uint64_t one = __ballot(internal && g == g0), has1 = __ballot((c & 1u) != 0), has2 = __ballot((c & 2u) != 0);
    const uint32_t a = (uint32_t)(__popcll(one & has1) + 2 * __popcll(one & has2)),
                   b = (uint32_t)(__popcll(~one & has1) + 2 * __popcll(~one & has2));
    if (lane == 0) {
      if (a) atomicAdd(groups + g0, a);
      if (b) atomicAdd(groups + g0 + 1, b);
    }
  }
  return total;
}

__device__ __forceinline__ void number_info(const Sah& s, uint32_t* __restrict__ info, uint32_t total) {
  info[RK_INFO_NODE_COUNT] = total;
  info[RK_INFO_FLAGS] |= s.ctl[kCtlFlags];
}

// A level, kNumberItems items per workgroup, after the groups before it; their
// internal items were counted when the level's queue was written. Clears the
// groups of the level after the next.
__global__ __launch_bounds__(1024) void k_sah_number(Sah s, uint32_t level, uint32_t m, uint32_t id0, uint32_t child0,
                                                     Node* __restrict__ nodes, uint32_t nodes_cap,
                                                     uint32_t* __restrict__ info, uint32_t total) {
  __shared__ uint32_t s_wave[16], s_tmp[16];
  const uint32_t* now = s.groups + (level % 3u) * s.group_cap;
  uint32_t* next = s.groups + ((level + 1u) % 3u) * s.group_cap;
  uint32_t* after = s.groups + ((level + 2u) % 3u) * s.group_cap;
  for (uint32_t i = blockIdx.x * 1024 + threadIdx.x; i < s.group_cap; i += gridDim.x * 1024) after[i] = 0u;
  uint32_t before = 0, before_total;
  for (uint32_t h = threadIdx.x; h < blockIdx.x; h += 1024) before += now[h];
  block_excl_scan(before, s_tmp, &before_total, 1024);
  const uint32_t* q_in = level & 1u ? s.q1 : s.q0;
  uint32_t* q_out = level & 1u ? s.q0 : s.q1;
  number_items(s, level, blockIdx.x * kNumberItems + threadIdx.x, m, q_in, q_out, id0, before_total, child0, next,
               nodes, nodes_cap, s_wave);
  if (info && blockIdx.x == 0 && threadIdx.x == 0) number_info(s, info, total);
}

// Levels [level, end) of at most 1024 items each, in one workgroup.
__global__ __launch_bounds__(1024) void k_sah_number_run(Sah s, uint32_t level, uint32_t end, uint32_t m, uint32_t id0,
                                                         uint32_t child0, Node* __restrict__ nodes, uint32_t nodes_cap,
                                                         uint32_t* __restrict__ info, uint32_t total) {
  __shared__ uint32_t s_wave[2][16];
  __shared__ uint32_t s_q[2][1024];
  uint32_t* next = s.groups + (end % 3u) * s.group_cap;
  uint32_t* after = s.groups + ((end + 1u) % 3u) * s.group_cap;
  for (uint32_t i = threadIdx.x; i < s.group_cap; i += 1024) next[i] = after[i] = 0u;
  if (info && threadIdx.x == 0) number_info(s, info, total);
  if (level && threadIdx.x < (m + 1) / 2) s_q[level & 1u][threadIdx.x] = (level & 1u ? s.q1 : s.q0)[threadIdx.x];
  __syncthreads();
  for (; level < end; ++level) {
    const bool last = level + 1 == end;
    uint32_t* q_out = last ? (level & 1u ? s.q0 : s.q1) : s_q[(level & 1u) ^ 1u];
    const uint32_t found = number_items(s, level, threadIdx.x, m, s_q[level & 1u], q_out, id0, 0, child0,
                                        last ? next : nullptr, nodes, nodes_cap, s_wave[level & 1u]);
    id0 = child0;
    m = 2 * found;
    child0 += m;
    __syncthreads();
  }
}

// The groups of the starting items, and the next two levels' cleared.
__global__ __launch_bounds__(1024) void k_sah_number_start(Sah s, uint32_t m) {
  __shared__ uint32_t s_sum;
  const uint32_t i = blockIdx.x * kNumberItems + threadIdx.x;
  if (threadIdx.x == 0) s_sum = 0u;
  for (uint32_t j = i; j < 2 * s.group_cap; j += gridDim.x * 1024) s.groups[s.group_cap + j] = 0u;
  __syncthreads();
  const uint64_t mask = __ballot(i < m && s.link[2 * (size_t)s.n + i] != kLeaf);
  if ((threadIdx.x & 63) == 0) atomicAdd(&s_sum, (uint32_t)__popcll(mask));
  __syncthreads();
  if (threadIdx.x == 0) s.groups[blockIdx.x] = s_sum;
}

// The faces' boxes, ids and a copy of them, and a large root's centroid bounds:
// kBoxPer faces per thread, so that few workgroups add to the same words.
constexpr uint32_t kBoxThreads = 1024, kBoxPer = 4;
__global__ __launch_bounds__(kBoxThreads) void k_boxes_root(Sah s, const uint4* __restrict__ faces,
                                                            const float4* __restrict__ verts, Box* __restrict__ boxes,
                                                            uint4* __restrict__ copy) {
  int b[6] = {f2o(RK_HUGE), f2o(RK_HUGE), f2o(RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE), f2o(-RK_HUGE)};
  uint4 f[kBoxPer];
#pragma unroll
  for (uint32_t u = 0; u < kBoxPer; ++u) {
    const uint32_t k = (blockIdx.x * kBoxPer + u) * kBoxThreads + threadIdx.x;
    f[u] = k < s.n ? faces[k] : make_uint4(0u, 0u, 0u, 0u);
  }
#pragma unroll
  for (uint32_t u = 0; u < kBoxPer; ++u) {
    const uint32_t k = (blockIdx.x * kBoxPer + u) * kBoxThreads + threadIdx.x;
    if (k >= s.n) continue;
    const float4 v0 = verts[f[u].x], v1 = verts[f[u].y], v2 = verts[f[u].z];
    Box x;
    x.mn = rk::min4(rk::min4(v0, v1), v2);
    x.mx = rk::max4(rk::max4(v0, v1), v2);
    float4* o = reinterpret_cast<float4*>(boxes + k);
    o[0] = x.mn;
    o[1] = x.mx;
    s.ids0[k] = k;
    copy[k] = f[u];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int c = f2o(center_axis(x, q));
      b[q] = min(b[q], c);
      b[3 + q] = max(b[3 + q], c);
    }
  }
  // a root of at most kChunk faces is k_sah_subtrees': big_cap is 0, and there are no bounds
  if (s.n > kChunk) add_bounds(b, s.bnd1);
}

__global__ __launch_bounds__(256) void k_gather_faces2(const uint4* __restrict__ src, const uint32_t* __restrict__ idx,
                                                       uint4* __restrict__ dst, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}
__global__ __launch_bounds__(256) void k_copy_faces2(const uint4* __restrict__ src, uint4* __restrict__ dst, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

}  // namespace

extern "C" size_t rk_build_sah_workspace_size(uint32_t face_count, uint32_t existing_nodes) {
  size_t n = face_count ? face_count : 1;
  size_t m = n + existing_nodes + 1;
  size_t big = n / kChunk + 1;
  size_t T = n / kChunk + big + 1;
  size_t b = 0;  // more than rk_build_sah takes
  b += rk_align_up(m * 48) * 2;
  b += rk_align_up(m * 4);
  b += rk_align_up(big * 3776);
  b += rk_align_up(m * 80);
  b += rk_align_up(T * 4) * 3;
  b += rk_align_up(n * 4);
  b += rk_align_up(n * 16);
  b += rk_align_up(128);
  b += rk_align_up((m / 1024 + 1) * 4);
  return b + 4096;
}

// void CUDA_buildMeshTreeSAH(CUDAMesh*, CUDAMeshTree*), CUDAMeshTree.cpp:34-38 /
// CUDA_buildMeshTreeSAH.cu:672-789. existing_nodes == 0: boxes and indices are
// (re)computed and the root is the mesh hitbox; existing_nodes > 0 (Hybrid):
// boxes/indices come from the LBVH pass and every leaf among nodes[0,
// existing_nodes) is refined. Faces are reordered by the final indices.
// Synchronises 'stream' a few times (once the levels that n faces cannot do
// without are queued, then once per two levels of big items, then for the level
// sizes); the node records and the info words are queued on 'stream' when it
// returns.
extern "C" rk_status rk_build_sah(rk_stream stream, rk_uint4* faces, const rk_float4* vertices, uint32_t face_count,
                                  const rk_aabox* hitbox, rk_aabox* boxes, uint32_t* indices, rk_bvnode* nodes,
                                  uint32_t existing_nodes, uint32_t nodes_capacity, uint32_t* info, void* ws,
                                  size_t ws_bytes) {
  const uint32_t n = face_count;
  if (n == 0 || !faces || !vertices || !hitbox || !boxes || !indices || !nodes || !info) return RK_ERROR_INVALID_VALUE;
  if (n >= (1u << 30)) return RK_ERROR_UNSUPPORTED;
  if ((size_t)nodes_capacity < (size_t)existing_nodes + 2 * (size_t)n - 1) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  Sah s;
  s.n = n;
  s.m_cap = (size_t)n + existing_nodes + 1;
  s.big_cap = n > kChunk ? n / kChunk + 1 : 0;
  s.chunks_cap = n > kChunk ? n / kChunk + s.big_cap + 1 : 0;
  s.group_cap = (uint32_t)(s.m_cap / kNumberItems + 1);
  s.boxes = reinterpret_cast<const Box*>(boxes);
  const size_t starts = existing_nodes ? existing_nodes : 1;
  const size_t spare = 4096 + rk_align_up((s.m_cap / 1024 + 1) * 4) - (s.m_cap / 1024 + 1) * 4;
  if (ws_bytes < rk_build_sah_workspace_size(n, existing_nodes) - spare) return RK_ERROR_WORKSPACE;
  RkArena ar(ws, ws_bytes);
  s.ids0 = indices;
  s.ids1 = ar.take<uint32_t>(n);
  s.rec = ar.take<Rec>(2 * (size_t)n + starts);
  s.link = ar.take<uint32_t>(2 * (size_t)n + starts);
  s.node0 = ar.take<uint32_t>(starts);
  s.q0 = ar.take<uint32_t>(2 * (size_t)n);
  s.roots = ar.take<uint2>(kClasses * s.m_cap);
  s.big0 = ar.take<BigItem>(2 * (size_t)s.big_cap);
  s.dec = ar.take<BigDec>(s.big_cap);
  s.chunk_item0 = ar.take<uint32_t>(2 * (size_t)s.chunks_cap);
  s.acc = ar.take<int>((size_t)s.big_cap * kAccWords);
  s.bnd0 = ar.take<int>((size_t)s.big_cap * 4 * kBoundWords);
  s.cum = ar.take<uint16_t>((size_t)kBins * s.chunks_cap);
  s.bin = ar.take<uint8_t>(n);
  s.ctl = ar.take<uint32_t>(ctl_words(n));
  s.groups = ar.take<uint32_t>(3 * (size_t)s.group_cap);
  uint4* ftmp = ar.take<uint4>(n);
  if (!s.ids1 || !s.rec || !s.link || !s.node0 || !s.q0 || !s.roots || !s.big0 || !s.dec || !s.chunk_item0 || !s.acc ||
      !s.bnd0 || !s.cum || !s.bin || !s.ctl || !s.groups || !ftmp)
    return RK_ERROR_WORKSPACE;
  s.q1 = s.q0 + n;
  s.big1 = s.big0 + s.big_cap;
  s.chunk_item1 = s.chunk_item0 + s.chunks_cap;
  s.bnd1 = s.bnd0 + (size_t)s.big_cap * 2 * kBoundWords;

  const bool root = existing_nodes == 0;
  const float4 rmin = make_float4(hitbox->min.x, hitbox->min.y, hitbox->min.z, hitbox->min.w);
  const float4 rmax = make_float4(hitbox->max.x, hitbox->max.y, hitbox->max.z, hitbox->max.w);
  hipLaunchKernelGGL(k_sah_clear, dim3(std::min(1024u, s.big_cap + 1)), dim3(256), 0, st, s, info, root ? 1 : 0,
                     rmin, rmax);
  RK_CHECK_LAUNCH();
  uint4* f = reinterpret_cast<uint4*>(faces);
  const unsigned per_face = (n + 255) / 256;
  constexpr uint32_t kHistRead = 64;  // levels read at once
  uint32_t got[kCtlHist + kHistRead] = {};
  auto read_ctl = [&](size_t words) -> rk_status {
    RK_HIP(hipMemcpyAsync(got, s.ctl, std::min(words, ctl_words(n)) * 4, hipMemcpyDeviceToHost, st));
    RK_HIP(hipStreamSynchronize(st));
    return RK_SUCCESS;
  };
  rk_status e;
  // big: items of more than kChunk faces on the level, or a bound of them; ahead:
  // levels to queue before the count is read back. A level has at most twice the
  // big items of the one before, and every kernel reads the exact counts on the
  // device, so a grid sized by a bound is only larger than needed. An item takes
  // as many levels of big items as it takes halvings down to kChunk, and seldom
  // more than two beyond; k_sah_subtrees is queued after those without a look, and
  // again for what further levels leave. (Read back before it too: 50 us more per
  // build.)
  uint32_t big, ahead = 2, starts_found = 1, largest = n;
  const uint32_t big_bound = n / (kChunk + 1);
  if (root) {
    hipLaunchKernelGGL(k_boxes_root, dim3((n + kBoxPer * kBoxThreads - 1) / (kBoxPer * kBoxThreads)), dim3(kBoxThreads),
                       0, st, s, f, reinterpret_cast<const float4*>(vertices), reinterpret_cast<Box*>(boxes), ftmp);
    RK_CHECK_LAUNCH();
    big = n > kChunk ? 1u : 0u;
  } else {
    hipLaunchKernelGGL(k_sah_init_from_leaves, dim3(1), dim3(1024), 0, st, s, reinterpret_cast<const Node*>(nodes),
                       existing_nodes);
    hipLaunchKernelGGL(k_copy_faces2, dim3(per_face), dim3(256), 0, st, f, ftmp, n);
    RK_CHECK_LAUNCH();
    if ((e = read_ctl(kCtlRead)) != RK_SUCCESS) return e;
    big = got[kCtlBig(0)];
    starts_found = big + got[kCtlRoots] + got[kCtlRoots + 1] + got[kCtlRoots + 2];
    largest = got[kCtlLargest];
  }
  for (uint32_t x = largest; x > kChunk; x -= x / 2) ++ahead;
  RootsDone done = {};
  uint32_t level = 0;
  do {
    for (uint32_t x = 0; x < ahead && big; ++x, ++level) {
      if (level > kLevelMax) return RK_ERROR_LAUNCH;
      const uint32_t par = level & 1u;
      const unsigned grid = n / kChunk + std::min(big, big_bound) + 1;  // chunks: see chunks_cap
      if (level == 0 && !root) hipLaunchKernelGGL(k_sah_bounds, dim3(grid), dim3(kCT), 0, st, s);
      hipLaunchKernelGGL(k_sah_bins, dim3(grid), dim3(kCT), 0, st, s, par);
      hipLaunchKernelGGL(k_sah_split, dim3((big + kSplitItems - 1) / kSplitItems), dim3(32 * kSplitItems), 0, st, s,
                         par, level);
      hipLaunchKernelGGL(k_sah_scatter, dim3(grid), dim3(kCT), 0, st, s, par);
      RK_CHECK_LAUNCH();
      big = std::min(2 * big, big_bound);
    }
    // 8 starting items a workgroup: starts of a face or two make more groups than
    // n / 256 (hybrid build from 1,280 leaves of one face 111 us with 6 workgroups,
    // 102 with 161; from 300,000 faces at depth 24 208 and 192)
    const uint32_t groups = std::max(n / 256, starts_found / 8) + 1;
    hipLaunchKernelGGL(k_sah_subtrees, dim3(std::min(2048u, groups)), dim3(kTreeThreads), 0, st, s, done);
    RK_CHECK_LAUNCH();
    if ((e = read_ctl(kCtlHist + kHistRead)) != RK_SUCCESS) return e;
    big = level ? got[kCtlBig(level & 1u)] : 0u;
    for (uint32_t c = 0; c < kClasses; ++c) done.n[c] = got[kCtlRoots + c];
    ahead = 2;
  } while (big);
  if (got[kCtlDeep]) return RK_ERROR_LAUNCH;  // refused: the faces stay as they are
  // CUDA_reorderMeshFaces, :778-784
  hipLaunchKernelGGL(k_gather_faces2, dim3(per_face), dim3(256), 0, st, ftmp, indices, f, n);
  RK_CHECK_LAUNCH();
  // the numbering, by the levels' sizes
  uint32_t hist[kLevelMax + 2] = {};  // (not from the heap, whose exceptions a C entry must not let out)
  std::copy_n(got + kCtlHist, kHistRead, hist);
  if (hist[kHistRead - 1]) {
    RK_HIP(hipMemcpyAsync(hist, s.ctl + kCtlHist, (ctl_words(n) - kCtlHist) * 4, hipMemcpyDeviceToHost, st));
    RK_HIP(hipStreamSynchronize(st));
  }
  const uint32_t total =
      (root ? 1u : existing_nodes) + 2u * std::accumulate(std::begin(hist), std::end(hist), 0u);
  Node* nd = reinterpret_cast<Node*>(nodes);
  uint32_t m = starts_found, id0 = 0, child0 = root ? 1u : existing_nodes;
  if (m > kNumberItems) {
    hipLaunchKernelGGL(k_sah_number_start, dim3((m + kNumberItems - 1) / kNumberItems), dim3(1024), 0, st, s, m);
    RK_CHECK_LAUNCH();
  }
  level = 0;
  do {  // level 0 writes the info words too, also with nothing on it
    uint32_t end = level + 1;
    uint32_t* out = level == 0 ? info : nullptr;
    if (m <= kNumberItems) {
      while (hist[end - 1] && 2 * hist[end - 1] <= kNumberItems) ++end;
      hipLaunchKernelGGL(k_sah_number_run, dim3(1), dim3(1024), 0, st, s, level, end, m, id0, child0, nd,
                         nodes_capacity, out, total);
    } else {
      hipLaunchKernelGGL(k_sah_number, dim3((m + kNumberItems - 1) / kNumberItems), dim3(1024), 0, st, s, level, m,
                         id0, child0, nd, nodes_capacity, out, total);
    }
    RK_CHECK_LAUNCH();
    for (; level < end; ++level) {
      id0 = child0;
      m = 2 * hist[level];
      child0 += m;
    }
  } while (m);
  return RK_SUCCESS;
}
