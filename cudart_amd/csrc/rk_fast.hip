// The throughput tree: a Morton LBVH built entirely on the GPU and a
// closest-hit traversal tuned for gfx950. No reference counterpart (the
// reference trees stop at tree_depth with leaves of up to 224 triangles); the
// triangle test is the reference's (CUDA_raytraceMeshTree.cu:57-89), so a
// hit's t, u, v are bit-identical to the reference's for the same triangle.
//
// Build:
//   k_fast_prep     per-face box (API array) and 30/63-bit Morton key
//   radix sort      (key, face) pairs
//   k_fast_hierarchy  topology, node boxes and leaf-ordered triangle records
//                     (v0, v1-v0, v2-v0; 48 B) bottom-up (agglomerative
//                     LBVH, Apetrei 2014) for the splits inside each
//                     512-position chunk; subtrees of <= leaf_max faces
//                     become leaves
//   k_hier_reduce     the same over the subtrees that 64 chunks left over,
//                     again until one group is left
//
// Node record (64 B): float4 (c0.lo.x, c0.hi.x, c0.lo.y, c0.hi.y),
//                     float4 (c1.lo.x, c1.hi.x, c1.lo.y, c1.hi.y),
//                     float4 (c0.lo.z, c0.hi.z, c1.lo.z, c1.hi.z),
//                     uint4  (ref0, ref1, count0, count1)
// ref: node index, or kLeafBit | first << 4 | (count - 1). The root is
// record 0 (a batch mesh's root: its first position); a node covering sorted
// positions [l, r] is record r when it is its parent's left child and record
// l when it is the right child, so the children of the split between p and
// p + 1 are records p and p + 1. n records for n faces.
#include <mutex>

#include "rk_device.h"
#include "rk_sort.h"

namespace {

using rk::Box;

constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kMaxLeaf = 16;

struct FNode { float4 a, b, c; uint4 d; };
static_assert(sizeof(FNode) == 64, "fast node is 64 B");

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}
__device__ __forceinline__ uint64_t spread21(uint64_t v) {
  v &= 0x1FFFFFull;
  v = (v | (v << 32)) & 0x1F00000000FFFFull;
  v = (v | (v << 16)) & 0x1F0000FF0000FFull;
  v = (v | (v << 8)) & 0x100F00F00F00F00Full;
  v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
  v = (v | (v << 2)) & 0x1249249249249249ull;
  return v;
}

// Per-face box (API array), Morton key and index. kPasses > 0: also counts the
// digits of the sort's kPasses passes (counts and info are zero already);
// otherwise it clears the build's info words. 'per' faces per thread.
constexpr uint32_t kPrepThreads = 1024;
constexpr uint32_t kCountInPrep = 1u << 21;
constexpr uint32_t kCountPer4 = 1u << 18;  // 4 faces per thread from here on: below, that leaves most CUs idle
template <typename K, int kPasses>
__global__ __launch_bounds__(kPrepThreads) void k_fast_prep(const uint4* __restrict__ faces,
                                                            const float4* __restrict__ verts, uint32_t n, float4 rmin,
                                                            float4 rmax, Box* __restrict__ boxes,
                                                            K* __restrict__ keys, uint32_t* __restrict__ vals,
                                                            uint32_t* __restrict__ info, uint32_t per,
                                                            uint32_t* __restrict__ counts, uint32_t copies) {
  constexpr int kWords = kPasses * 256;
  __shared__ uint32_t s_hist[kWords ? kWords : 1];
  if (kPasses) {
    for (int i = threadIdx.x; i < kWords; i += kPrepThreads) s_hist[i] = 0u;
    __syncthreads();
  } else if (blockIdx.x == 0 && threadIdx.x < RK_INFO_WORDS) {
    info[threadIdx.x] = 0u;
  }
  const float4 len = rk::sub4(rmax, rmin);
  const float cells = sizeof(K) == 4 ? 1024.0f : 2097152.0f;
  const uint32_t top = sizeof(K) == 4 ? 1023u : 2097151u;
  const float sx = cells / len.x, sy = cells / len.y, sz = cells / len.z;
  const size_t base = (size_t)blockIdx.x * per * kPrepThreads + threadIdx.x;
  for (uint32_t u = 0; u < per; ++u) {
    const size_t kk = base + (size_t)u * kPrepThreads;
    if (kk >= n) break;
    const uint32_t k = (uint32_t)kk;
    const uint4 f = faces[k];
    const float4 v0 = verts[f.x], v1 = verts[f.y], v2 = verts[f.z];
    Box b;
    b.mn = rk::min4(rk::min4(v0, v1), v2);
    b.mx = rk::max4(rk::max4(v0, v1), v2);
    if (boxes) {  // the API's per-face boxes, when the caller keeps them
      float4* o = reinterpret_cast<float4*>(boxes + k);
      o[0] = b.mn;
      o[1] = b.mx;
    }
    const float4 c = rk::muls4(rk::add4(b.mn, b.mx), 0.5f);
    const uint32_t qx = min(rk::f2u_sat((c.x - rmin.x) * sx), top);
    const uint32_t qy = min(rk::f2u_sat((c.y - rmin.y) * sy), top);
    const uint32_t qz = min(rk::f2u_sat((c.z - rmin.z) * sz), top);
    K key;
    if (sizeof(K) == 4) key = (K)((spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz));
    else key = (K)((spread21(qx) << 2) | (spread21(qy) << 1) | spread21(qz));
    keys[k] = key;
    vals[k] = k;
    if (kPasses) rk_count_digits<K, kPasses>(s_hist, key);
  }
  if (kPasses) {
    __syncthreads();
    rk_flush_digits<kPasses, (int)kPrepThreads>(s_hist, counts, copies);
  }
}

// Split key between sorted positions i and i+1 (Apetrei 2014, "Fast and
// simple agglomerative LBVH construction"): the XOR of the two Morton keys,
// with the top bit set so that any difference in the keys outranks the index
// tie-break used for equal keys (the XOR of the two positions). Larger means
// the two positions separate higher in the tree. Two splits that bound the
// same node never compare equal.
template <typename K>
__device__ __forceinline__ uint64_t split_key(const K* __restrict__ keys, uint32_t i) {
  const uint64_t x = (uint64_t)(keys[i] ^ keys[i + 1]);
  return x ? (x | 0x8000000000000000ull) : (uint64_t)(i ^ (i + 1));
}

// Outward padding: a relative 2^-18 of the coordinate magnitude plus the same
// fraction of the extent, so every box contains what the triangle test can
// accept inside it despite rounding on either side.
__device__ __forceinline__ void pad_box(float& lo, float& hi) {
  float m = rk::fmx(fabsf(lo), fabsf(hi));
  float e = hi - lo;
  float p = (m + e) * 3.814697265625e-06f + 1e-30f;
  lo = lo - p;
  hi = hi + p;
}

// A finished subtree as its sibling sees it: box (unpadded), reference, and
// the end of its range that the sibling does not know: the item, its position
// and the split key beyond it.
struct alignas(16) Part {
  float lox, loy, loz, hix, hiy, hiz;
  uint32_t ref, end;
  uint64_t key;
  uint32_t pos, pad;
};
static_assert(sizeof(Part) == 48, "part is 48 B");
__device__ __forceinline__ void write_node(FNode* __restrict__ nodes, uint32_t idx, const Part& c0, const Part& c1,
                                           uint32_t n0, uint32_t n1) {
  float a0 = c0.lox, a1 = c0.hix, a2 = c0.loy, a3 = c0.hiy, a4 = c0.loz, a5 = c0.hiz;
  float b0 = c1.lox, b1 = c1.hix, b2 = c1.loy, b3 = c1.hiy, b4 = c1.loz, b5 = c1.hiz;
  pad_box(a0, a1); pad_box(a2, a3); pad_box(a4, a5);
  pad_box(b0, b1); pad_box(b2, b3); pad_box(b4, b5);
  FNode* p = nodes + idx;
  p->a = make_float4(a0, a1, a2, a3);
  p->b = make_float4(b0, b1, b2, b3);
  p->c = make_float4(a4, a5, b4, b5);
  p->d = make_uint4(c0.ref, c1.ref, n0, n1);
}

#ifndef RK_HIER_THREADS
#define RK_HIER_THREADS 512
#endif
constexpr uint32_t kChunk = RK_HIER_THREADS;  // sorted positions per workgroup of k_fast_hierarchy, one per thread

__device__ __forceinline__ Part merge_parts(const Part& lc, const Part& rc) {
  Part up;
  up.lox = rk::fmn(lc.lox, rc.lox);
  up.loy = rk::fmn(lc.loy, rc.loy);
  up.loz = rk::fmn(lc.loz, rc.loz);
  up.hix = rk::fmx(lc.hix, rc.hix);
  up.hiy = rk::fmx(lc.hiy, rc.hiy);
  up.hiz = rk::fmx(lc.hiz, rc.hiz);
  return up;
}

// Parent of the subtree [l, r]: the split at r when split_key(r) <
// split_key(l - 1) (the subtree is its left child), else the split at l - 1.
__device__ __forceinline__ bool left_of_parent(bool has_l, bool has_r, uint64_t kl, uint64_t kr) {
  return !has_l || (has_r && kr < kl);
}

// The hierarchy, bottom-up (agglomerative LBVH, Apetrei 2014): a subtree
// covering sorted positions [l, r] is a child of the split at r or at l - 1,
// whichever has the smaller split key; of the two subtrees that arrive at a
// split, the second has it merged. This gives the binary radix tree of Karras
// 2012 without per-node binary searches.
//
// A workgroup takes a run of up to kT consecutive items (single positions in
// k_fast_hierarchy, subtrees left over by earlier passes in k_hier_reduce),
// one per thread, and exchanges through LDS alone. A split whose range lies
// inside the run sees both children arrive; at any other at most one does, and
// that subtree is left over for the next pass. The splits that cross one end
// of the run are nested, so at most two subtrees per level of the tree are
// left over; 10 to 12 per 512 positions on the meshes measured.
//
// Merges run in rounds: a round merges the splits in a queue, one per thread,
// and those whose parents become ready fill the next round's queue. Once at
// most 64 are ready they fit the first wave, whose lanes go on alone, without
// queue or barriers, each with its subtree in registers. What bounds the pass
// is issuing the merges: a thread that climbed on by itself from its leaf left
// its wave with a few active lanes for a dozen steps (80 wave-steps per 512
// positions against about 20), and the splits that cross chunks took three
// round trips to memory per level. On the 1M-face terrain the passes took 111
// us that way.
//
// Slots: a subtree on items [a, b] waits for its sibling in slot b of part as
// a left child and in slot a as a right child, so the children of split q
// (between items q - 1 and q) are in slots q - 1 and q; end is the item at the
// subtree's other end. Slots a..b belong to that subtree alone.

// A subtree that a run left over, for the next pass: its part, its positions
// [l, r] and the split key after r.
struct HierItem {
  float4 a, b, c;  // (lo.xyz, hi.x), (hi.yz, ref, l), (r, 0, key)
};
static_assert(sizeof(HierItem) == 48, "item is 48 B");

constexpr uint32_t kFromLeft = 1u, kFromRight = 2u;  // HierLds::flag: the children that have arrived

template <uint32_t kT>
struct HierLds {
  Part part[kT];
  uint64_t key[kT + 1];   // key[q]: the split key before item q; key[m] after the last; ~0 past the array's ends
  uint32_t first[kT], last[kT];  // item k's positions
  uint32_t flag[kT + 1];  // split q's arrivals
  uint32_t cnt[3];        // entries of the rounds' queues
  uint32_t wcnt[kT / 64];
  uint16_t queue[2][kT / 2];
};

// Whether a key separates two meshes of a batch (or is past an end): keys are
// mesh << 30 | 30-bit code, so the XOR reaches bit 30.
__device__ __forceinline__ bool between_meshes(uint64_t key) { return ((key << 1) >> 31) != 0ull; }

// A subtree on items [a, b] and positions [l, r], with the split keys before
// and after it.
struct Sub {
  Part p;  // box and reference
  uint32_t a, b, l, r;
  uint64_t kl, kr;
};

// The subtree u goes to its parent, split q (left: as the left child); the
// children that had arrived there before.
template <uint32_t kT>
__device__ __forceinline__ uint32_t hier_arrive(HierLds<kT>& s, Sub& u, uint32_t n, bool& left, uint32_t& q) {
  left = left_of_parent(u.l > 0u, u.r + 1u < n, u.kl, u.kr);
  q = left ? u.b + 1u : u.a;
  u.p.end = left ? u.a : u.b;
  u.p.pos = left ? u.l : u.r;
  u.p.key = left ? u.kl : u.kr;
  s.part[left ? u.b : u.a] = u.p;
  // a wave's LDS accesses keep their order, which is all the first wave's
  // going on alone needs; between waves there is a barrier
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  const uint32_t before = __hip_atomic_fetch_add(&s.flag[q], left ? kFromLeft : kFromRight, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return before;
}

// Merges split q's children lc and rc into u, whose range is set: the split's
// record is written unless it collapses into a leaf (p: the left child's last
// position), and u goes to its parent. True when that is ready too.
template <uint32_t kT, bool kBatch>
__device__ __forceinline__ bool hier_merge(HierLds<kT>& s, uint32_t n, uint32_t leaf_max, FNode* __restrict__ nodes,
                                           const Part& lc, const Part& rc, uint32_t p, Sub& u, bool& left,
                                           uint32_t& q) {
  const bool root = kBatch ? between_meshes(u.kl) && between_meshes(u.kr) : u.l == 0u && u.r + 1u == n;
  const uint32_t cnt = u.r - u.l + 1u;
  uint32_t before = 0u, idx = u.l;  // a root's record goes to its first position
  u.p = merge_parts(lc, rc);
  if (!root) {
    // any other to its last position as a left child and to its first as a
    // right child: the children of the split between p and p + 1 are then
    // records p and p + 1 (Karras 2012's numbering)
    if (left_of_parent(u.l > 0u, u.r + 1u < n, u.kl, u.kr)) idx = u.r;
    u.p.ref = cnt <= leaf_max ? (kLeafBit | (u.l << 4) | (cnt - 1u)) : idx;
    before = hier_arrive(s, u, n, left, q);
  }
  if (root || cnt > leaf_max) write_node(nodes, idx, lc, rc, p - u.l + 1u, u.r - p);
  return before != 0u;
}

// Completes the run's splits: every first arrival is in (ready, q: this
// thread's second one), keys and zeroed flags since a barrier. Ends with one.
template <uint32_t kT, bool kBatch>
__device__ __forceinline__ void hier_rounds(HierLds<kT>& s, uint32_t n, uint32_t leaf_max, FNode* __restrict__ nodes,
                                            bool ready, uint32_t q) {
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  auto push = [&](bool sec, uint32_t sq, uint32_t qi, uint32_t ci) {
    const uint64_t mask = __ballot(sec);
    if (mask == 0ull) return;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(&s.cnt[ci], (uint32_t)__popcll(mask));
    base = __builtin_amdgcn_readfirstlane(base);
    if (sec) s.queue[qi][base + (uint32_t)__popcll(mask & rk::lanemask_lt())] = (uint16_t)sq;
  };
  // split sq's children and range; the left child's last position
  auto load = [&](uint32_t sq, Part& lc, Part& rc, Sub& u) {
    lc = s.part[sq - 1u];
    rc = s.part[sq];
    u.a = lc.end;
    u.b = rc.end;
    u.l = lc.pos;
    u.r = rc.pos;
    u.kl = lc.key;
    u.kr = rc.key;
    return s.last[sq - 1u];
  };
  push(ready, q, 0u, 0u);
  for (uint32_t r = 0;; ++r) {
    __syncthreads();
    const uint32_t cnt = s.cnt[r % 3u];
    if (cnt <= 64u) {
      if (w == 0 && lane < cnt) {
        Part lc, rc;
        Sub u;
        bool left;
        uint32_t p = load(s.queue[r & 1u][lane], lc, rc, u);
        while (hier_merge<kT, kBatch>(s, n, leaf_max, nodes, lc, rc, p, u, left, q)) {
          const Part sib = s.part[left ? q : q - 1u];
          p = left ? u.r : u.l - 1u;  // a split's children are next to each other
          lc = left ? u.p : sib;
          rc = left ? sib : u.p;
          u.a = left ? u.a : sib.end;
          u.l = left ? u.l : sib.pos;
          u.kl = left ? u.kl : sib.key;
          u.b = left ? sib.end : u.b;
          u.r = left ? sib.pos : u.r;
          u.kr = left ? sib.key : u.kr;
        }
      }
      break;
    }
    if (t == 0) s.cnt[(r + 2u) % 3u] = 0u;  // last read in the round before
    // at most kT / 2 entries: two items each
    uint32_t nq = 0u;
    bool sec = false;
    if (t < cnt) {
      Part lc, rc;
      Sub u;
      bool left;
      const uint32_t p = load(s.queue[r & 1u][t], lc, rc, u);
      sec = hier_merge<kT, kBatch>(s, n, leaf_max, nodes, lc, rc, p, u, left, nq);
    }
    push(sec, nq, (r & 1u) ^ 1u, (r + 1u) % 3u);
  }
  __syncthreads();
}

// The left-over subtree that waits at split q, if one does.
struct Left {
  bool has;
  Part part;
  uint32_t l, r;  // positions
  uint64_t kl, kr;
};
template <uint32_t kT>
__device__ __forceinline__ Left left_over(const HierLds<kT>& s, uint32_t m, uint32_t q) {
  Left o;
  const uint32_t f = q <= m ? s.flag[q] : 0u;
  o.has = f == kFromLeft || f == kFromRight;
  o.l = o.r = 0u;
  o.kl = o.kr = 0ull;
  if (o.has) {
    const bool left = f == kFromLeft;
    o.part = s.part[left ? q - 1u : q];
    o.l = left ? o.part.pos : s.first[q];
    o.r = left ? s.last[q - 1u] : o.part.pos;
    o.kl = left ? o.part.key : s.key[q];
    o.kr = left ? s.key[q] : o.part.key;
  }
  return o;
}

// Ranks of the left-over subtrees of splits 0 .. kT - 1 (has: this thread's),
// and their number. Subtrees in item order wait at splits in increasing order.
template <uint32_t kT>
__device__ __forceinline__ uint32_t hier_rank(HierLds<kT>& s, bool has, uint32_t& total) {
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint64_t mask = __ballot(has);
  if (lane == 0) s.wcnt[w] = (uint32_t)__popcll(mask);
  __syncthreads();
  uint32_t before = (uint32_t)__popcll(mask & rk::lanemask_lt());
  total = 0u;
  for (uint32_t k = 0; k < kT / 64; ++k) {
    if (k < w) before += s.wcnt[k];
    total += s.wcnt[k];
  }
  return before;
}

__device__ __forceinline__ void store_item(HierItem* __restrict__ it, const Part& p, uint32_t l, uint32_t r,
                                           uint64_t key) {
  it->a = make_float4(p.lox, p.loy, p.loz, p.hix);
  it->b = make_float4(p.hiy, p.hiz, __uint_as_float(p.ref), __uint_as_float(l));
  it->c = make_float4(__uint_as_float(r), 0.0f, __uint_as_float((uint32_t)key), __uint_as_float((uint32_t)(key >> 32)));
}

// The chunk pass: kChunk consecutive sorted positions per workgroup, one per
// thread, whose triangle record it also writes. With kBatch the positions hold
// many meshes, sorted by (mesh, Morton code): keys are mesh << 30 | 30-bit
// code, so every split between two meshes ranks above every split inside one,
// and a subtree between two such splits is its mesh's root, whose record goes
// to the mesh's first position. Mesh m's nodes and triangle records then
// occupy [face_offset, face_offset + face_count).
template <typename K, bool kBatch>
__global__ __launch_bounds__(kChunk) void k_fast_hierarchy(const K* __restrict__ keys,
                                                           const uint32_t* __restrict__ order,
                                                           const uint4* __restrict__ faces,
                                                           const float4* __restrict__ verts, uint32_t n,
                                                           uint32_t leaf_max, FNode* __restrict__ nodes,
                                                           float4* __restrict__ tris,
                                                           const rk_batch_mesh* __restrict__ meshes,
                                                           HierItem* __restrict__ items,
                                                           uint32_t* __restrict__ counts) {
  __shared__ HierLds<kChunk> s;
  const uint32_t t = threadIdx.x;
  const uint32_t c0 = blockIdx.x * kChunk;
  const uint32_t m = min(kChunk, n - c0);
  const uint32_t i = c0 + t;
  // leaf loads first: their latency overlaps the split keys'
  uint32_t fid = 0;
  float4 v0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), v1 = v0, v2 = v0;
  if (t < m) {
    fid = order[i];
    uint32_t voff = 0;
    if (kBatch) voff = meshes[(uint32_t)((uint64_t)keys[i] >> 30)].vertex_offset;
    const uint4 f = faces[fid];
    v0 = verts[f.x + voff];
    v1 = verts[f.y + voff];
    v2 = verts[f.z + voff];
  }
  for (uint32_t k = t; k <= m; k += kChunk) {
    const int64_t x = (int64_t)c0 - 1 + (int64_t)k;
    s.key[k] = (x >= 0 && x + 1 < (int64_t)n) ? split_key(keys, (uint32_t)x) : ~0ull;
    s.flag[k] = 0u;
  }
  s.first[t] = s.last[t] = i;
  if (t < 3u) s.cnt[t] = 0u;
  __syncthreads();
  bool ready = false;
  uint32_t q = 0;
  if (t < m) {
    const float4 e1 = rk::sub4(v1, v0), e2 = rk::sub4(v2, v0);
    tris[3 * (size_t)i + 0] = make_float4(v0.x, v0.y, v0.z, __uint_as_float(fid));
    tris[3 * (size_t)i + 1] = make_float4(e1.x, e1.y, e1.z, 0.0f);
    tris[3 * (size_t)i + 2] = make_float4(e2.x, e2.y, e2.z, 0.0f);
    Sub u;
    u.a = u.b = t;
    u.l = u.r = i;
    u.kl = s.key[t];
    u.kr = s.key[t + 1u];
    Part& me = u.p;
    me.lox = rk::fmn(rk::fmn(v0.x, v1.x), v2.x);
    me.loy = rk::fmn(rk::fmn(v0.y, v1.y), v2.y);
    me.loz = rk::fmn(rk::fmn(v0.z, v1.z), v2.z);
    me.hix = rk::fmx(rk::fmx(v0.x, v1.x), v2.x);
    me.hiy = rk::fmx(rk::fmx(v0.y, v1.y), v2.y);
    me.hiz = rk::fmx(rk::fmx(v0.z, v1.z), v2.z);
    me.ref = kLeafBit | (i << 4);  // count - 1 = 0
    if (kBatch ? between_meshes(u.kl) && between_meshes(u.kr) : n == 1u) {
      // a single face: root with one leaf child and one empty child
      Part empty;
      empty.lox = empty.loy = empty.loz = RK_HUGE;
      empty.hix = empty.hiy = empty.hiz = -RK_HUGE;
      empty.ref = kLeafBit;
      write_node(nodes, i, me, empty, 1, 0);
    } else {
      bool left;
      ready = hier_arrive(s, u, n, left, q) != 0u;
    }
  }
  hier_rounds<kChunk, kBatch>(s, n, leaf_max, nodes, ready, q);
  const Left o = left_over(s, m, t);
  uint32_t total;
  const uint32_t rank = hier_rank(s, o.has, total);
  if (o.has) store_item(items + c0 + rank, o.part, o.l, o.r, o.kr);
  if (t == 0) {
    if (m == kChunk) {  // the split after the last item, which no thread above has
      const Left e = left_over(s, m, m);
      if (e.has) store_item(items + c0 + total++, e.part, e.l, e.r, e.kr);
    }
    counts[blockIdx.x] = total;
  }
}

// One group of up to kReduceFan runs, whose left-over subtrees (counts[c] of
// them from items[c * kChunk] on, c = the run's first chunk, every stride-th)
// become the items of one run, completed as above; what is left over goes to
// the group's first chunk. More items than threads are taken in steps, each
// with the subtrees the one before left over in front.
//
// 1024 threads take 128 VGPRs each, so the workgroup waits for a whole CU to fall
// free, which on a GPU full of another stream's traces takes as long as the traces
// (a served frame's pass: 188 us of waiting). Few enough runs (kReduceSmall chunks
// with about 12 subtrees each, kReduceSmallGroups groups with about 25) that 512
// threads take them in one step as fast have half of that: 32 requests served in
// 3.45 ms, with 1024 threads for all 3.58-3.74; with 512 for all the 1M-face build
// takes 180 us, not 158.
constexpr uint32_t kReduceFan = 64, kReduceSmall = 40, kReduceSmallGroups = 16;
template <typename K, bool kBatch, uint32_t kReduceThreads>
__global__ __launch_bounds__(kReduceThreads) void k_hier_reduce(const K* __restrict__ keys, uint32_t n,
                                                                uint32_t leaf_max, uint32_t chunks, uint32_t stride,
                                                                FNode* __restrict__ nodes,
                                                                HierItem* __restrict__ items,
                                                                uint32_t* __restrict__ counts) {
  constexpr uint32_t kT = kReduceThreads;
  static_assert(kReduceFan == 64, "one lane per run");
  __shared__ HierLds<kT> s;
  __shared__ uint32_t s_off[kReduceFan + 1];
  const uint32_t t = threadIdx.x;
  const uint32_t base = blockIdx.x * kReduceFan * stride;  // the group's first chunk
  uint64_t key0 = ~0ull;  // before the group's first position
  if (t == 0 && base > 0u) key0 = split_key(keys, base * kChunk - 1u);
  if (t < 64u) {
    const uint64_t c = (uint64_t)base + (uint64_t)t * stride;
    uint32_t incl = c < chunks ? counts[c] : 0u;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, 64);
      if (t >= (uint32_t)off) incl += y;
    }
    s_off[t + 1u] = incl;
    if (t == 0) s_off[0] = 0u;
  }
  __syncthreads();
  const uint32_t total = s_off[kReduceFan];
  uint32_t done = 0, m = 0, left = 0;  // items taken; items in front from the step before; left over
  for (;;) {
    const uint32_t take = min(total - done, kT - m);
    Sub u;
    u.a = u.b = t;
    if (t < m) {  // in place since the step before
      u.p = s.part[t];
      u.l = s.first[t];
      u.r = s.last[t];
    } else if (t < m + take) {
      const uint32_t e = done + t - m;
      uint32_t lo = 0, hi = kReduceFan - 1u;  // the last run with s_off <= e
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) >> 1;
        if (s_off[mid] <= e) lo = mid;
        else hi = mid - 1u;
      }
      const HierItem it = items[((size_t)base + (size_t)lo * stride) * kChunk + (e - s_off[lo])];
      u.p.lox = it.a.x; u.p.loy = it.a.y; u.p.loz = it.a.z; u.p.hix = it.a.w;
      u.p.hiy = it.b.x; u.p.hiz = it.b.y;
      u.p.ref = __float_as_uint(it.b.z);
      u.l = __float_as_uint(it.b.w);
      u.r = __float_as_uint(it.c.x);
      s.first[t] = u.l;
      s.last[t] = u.r;
      s.key[t + 1u] = (uint64_t)__float_as_uint(it.c.z) | ((uint64_t)__float_as_uint(it.c.w) << 32);
      // (a batch's first left-over subtree may lie further on)
      if (t == 0) s.key[0] = u.l == base * kChunk ? key0 : split_key(keys, u.l - 1u);
    }
    m += take;
    done += take;
    for (uint32_t k = t; k <= m; k += kT) s.flag[k] = 0u;
    if (t < 3u) s.cnt[t] = 0u;
    __syncthreads();
    bool ready = false, as_left;
    uint32_t q = 0;
    if (t < m) {
      u.kl = s.key[t];
      u.kr = s.key[t + 1u];
      ready = hier_arrive(s, u, n, as_left, q) != 0u;
    }
    hier_rounds<kT, kBatch>(s, n, leaf_max, nodes, ready, q);
    // split kT, which no thread has when m == kT, goes last
    const Left o = left_over(s, m, t);
    Left e;
    e.has = false;
    if (t == 0 && m == kT) e = left_over(s, m, m);
    const uint32_t rank = hier_rank(s, o.has, left);
    const uint32_t last = left;
    if (m == kT && (s.flag[kT] == kFromLeft || s.flag[kT] == kFromRight)) ++left;
    if (done == total || left >= kT) {  // left < kT: the tree's depth bounds it
      if (o.has) store_item(items + (size_t)base * kChunk + rank, o.part, o.l, o.r, o.kr);
      if (e.has) store_item(items + (size_t)base * kChunk + last, e.part, e.l, e.r, e.kr);
      if (t == 0) counts[base] = left;
      return;
    }
    // the left-over subtrees become the next step's first items
    __syncthreads();
    auto keep = [&](const Left& x, uint32_t at) {
      s.part[at] = x.part;
      s.first[at] = x.l;
      s.last[at] = x.r;
      s.key[at + 1u] = x.kr;
      if (at == 0u) s.key[0] = x.kl;
    };
    if (o.has) keep(o, rank);
    if (e.has) keep(e, last);
    m = left;
    __syncthreads();
  }
}

// ---- trace -------------------------------------------------------------------

// The traversal stack holds at most one entry per tree level, and a radix
// tree over b-bit keys with position tie-breaks (< 2^27 positions) is at most
// b + 27 levels deep: 57 for 30-bit keys, 90 for 63-bit keys.
#ifndef RK_TRACE_STACK
#define RK_TRACE_STACK 96
#endif
constexpr int kStack = RK_TRACE_STACK;
#ifndef RK_LDS_STACK
#define RK_LDS_STACK 8
#endif
// Stack entries per lane kept in LDS: 8 x 8 B x 64 lanes is 4 KB per wave, with the
// exchange words 4.5: frames have 24 waves per CU by their 80 registers, which leave
// room for 12 entries. Incoherent rays go deeper: 12 entries in batches (24 waves, or
// 20 by the queue kernel's 93 registers; 1024-mesh batch with 9, 12, 15, 19: 4.01,
// 3.96, 4.07, 4.09 ms) and sorted traces (86 registers, 20 waves; 9, 12 and 15 within
// 1%: 1M rays on the 100k soup 0.61 ms, 2M on 300k faces 1.78), 15, all that 20 waves
// leave room for, on trees past the L2 (16M sorted rays on the 10M soup with 12, 15
// and 19: 23.9, 23.9 and 24.6 ms).
constexpr int kLdsStack = RK_LDS_STACK, kDeepLdsStack = 12, kDeepestLdsStack = 15;

// intersectTriRay, CUDA_raytraceMeshTree.cu:57-89, with vert0.w = edge1.w =
// edge2.w = 0 (:174-176) and the reference's four-term dot products. eps is
// the reference's EPSILON (1e-6, :36) unless the caller chose another.
__device__ __forceinline__ bool tri_ray(float4 orig, float4 dir, float4 v0, float4 e1, float4 e2, float eps, float& t,
                                        float& u, float& v) {
  float4 pvec = rk::cross4(dir, e2);
  float det = rk::dot4(e1, pvec);
  if (det > -eps && det < eps) return false;
  float inv_det = 1.0f / det;
  float4 tvec = rk::sub4(orig, v0);
  u = rk::dot4(tvec, pvec) * inv_det;
  if (u < 0.0f || u > 1.0f) return false;
  float4 qvec = rk::cross4(tvec, e1);
  v = rk::dot4(dir, qvec) * inv_det;
  if (v < 0.0f || u + v > 1.0f) return false;
  t = rk::dot4(e2, qvec) * inv_det;
  return t >= 0.0f;
}

__device__ __forceinline__ float safe_inv(float d) {
  float a = fabsf(d) > 1e-20f ? d : (d < 0.0f ? -1e-20f : 1e-20f);
  return 1.0f / a;
}

// The slab test of a node record's two child boxes against a ray given by its
// inverse direction (ix, iy, iz) and origin terms (ox = o.x * ix, ...), over
// [0, bound]: entry distances and whether each box is hit.
struct Slab2 {
  float tmin0, tmin1;
  bool h0, h1;
};
__device__ __forceinline__ Slab2 slab2(const FNode& nd, float ix, float iy, float iz, float ox, float oy, float oz,
                                       float bound) {
  const float a0 = __builtin_fmaf(nd.a.x, ix, -ox), a1 = __builtin_fmaf(nd.a.y, ix, -ox);
  const float a2 = __builtin_fmaf(nd.a.z, iy, -oy), a3 = __builtin_fmaf(nd.a.w, iy, -oy);
  const float a4 = __builtin_fmaf(nd.c.x, iz, -oz), a5 = __builtin_fmaf(nd.c.y, iz, -oz);
  const float b0 = __builtin_fmaf(nd.b.x, ix, -ox), b1 = __builtin_fmaf(nd.b.y, ix, -ox);
  const float b2 = __builtin_fmaf(nd.b.z, iy, -oy), b3 = __builtin_fmaf(nd.b.w, iy, -oy);
  const float b4 = __builtin_fmaf(nd.c.z, iz, -oz), b5 = __builtin_fmaf(nd.c.w, iz, -oz);
  const float tmin0 = fmaxf(fmaxf(fminf(a0, a1), fminf(a2, a3)), fmaxf(fminf(a4, a5), 0.0f));
  const float tmax0 = fminf(fminf(fmaxf(a0, a1), fmaxf(a2, a3)), fminf(fmaxf(a4, a5), bound));
  const float tmin1 = fmaxf(fmaxf(fminf(b0, b1), fminf(b2, b3)), fmaxf(fminf(b4, b5), 0.0f));
  const float tmax1 = fminf(fminf(fmaxf(b0, b1), fmaxf(b2, b3)), fminf(fmaxf(b4, b5), bound));
  return Slab2{tmin0, tmin1, tmin0 <= tmax0, tmin1 <= tmax1};
}

// A traversal's result: the sorted position of the closest hit (~0: none),
// its t (the tmax it started with when there is no hit), u and v.
struct RayHit {
  uint32_t pos;
  float t, u, v;
};

// Closest hit of each lane's ray in the tree rooted at 'root' (positions and
// node records share one index space of n_tris). Depth-first, nearer child
// first; a pending child is skipped once the hit found is nearer than its
// entry point. Ties on t go to the smallest original face id, so the result
// does not depend on the tree or on the order of the visits.
//
// The wave shares the work. Every lane starts on its own ray (has_ray); a
// lane with nothing left to do takes the newest pending subtree of a lane
// that still has some (one per donor and step) and traverses it for that
// lane's ray, culling against the owner's best hit so far. A helper's best
// hit is merged into its owner's when the subtree is done, by (t, original
// id). A frame then waits less on its few long rays (grazing rays near a
// horizon), which would otherwise keep a wave running with one active lane.
// Every lane of the wave must call it; xchg is this wave's kXchgWords words of
// LDS.
//
// The stack: its first kLds entries live in LDS (lds: this workgroup's
// kLds x kWG entries, entry e of thread x at e * kWG + x), the rest in
// per-lane scratch. Pending entries rarely go deeper than a dozen or two, and
// an LDS access takes a fraction of the time of a scratch access that misses
// the L1 (the scratch of thousands of resident lanes does not fit in it).
// LDS words per wave for the exchange of pending subtrees: reference, entry
// distance, owner lane and donor lane of each donation. A step has at most 32: a
// lane is a donor or idle, not both.
constexpr int kXchg = 32, kXchgWords = 4 * kXchg;

// kOldest: a donor hands out its oldest pending entry (the bottom of its
// stack: the subtree nearest the root, the largest) instead of its newest, as
// a work-stealing deque does, so a helper gets more work and soon has pending
// entries of its own to hand on. The stack is then the range [sb, sp); it is
// reset to empty at [0, 0) whenever it drains, and an index still stands for
// one level of the current path, so sp stays within the depth bound.
//
// kLeafBatch > 0 postpones leaves: a lane that reaches a leaf keeps it as its
// one pending leaf and goes on to its next pending subtree, and the wave
// tests the pending leaves together once kLeafBatch lanes hold one (or a lane
// cannot go on without its leaf: it reached a second leaf, or its subtree is
// done). With one face per leaf some lane of a busy wave is at a leaf on
// almost every step, so testing leaves at once issues the triangle test on
// almost every step. A postponed leaf leaves the culling bound looser for a
// few steps, so a lane may visit a node it would have culled; the closest hit
// is the same. kDonateMin: the exchange runs only on steps where at least this
// many lanes are idle.
// The faces of leaf 'ref' against the job's ray (jo, jd). own: the ray is
// this lane's, and a hit goes to its best (o_*); otherwise to this helper's
// best (j_*), kept only if it can beat the owner's best as of this step (dmax,
// d_hit). Ties on t go to the smaller original id. A macro, not a function: the
// best-hit variables stay in registers only if no reference to them is taken.
#define RK_TRI_HIT(r0, e1, e2, position)                                                               \
  do {                                                                                                 \
    float4 v0 = r0;                                                                                    \
    v0.w = 0.0f;                                                                                       \
    float t, u, v;                                                                                     \
    if (kCount) ++n_tri;                                                                               \
    if (tri_ray(jo, jd, v0, e1, e2, eps, t, u, v)) {                                                   \
      const uint32_t oid = __float_as_uint((r0).w);                                                    \
      if (own) {                                                                                       \
        if (t < o_t || (o_pos != 0xFFFFFFFFu && t == o_t && oid < o_oid)) {                            \
          o_t = t; o_pos = (position); o_oid = oid; o_u = u; o_v = v;                                  \
        }                                                                                              \
      } else if ((t < dmax || (d_hit && t == dmax)) &&                                                 \
                 (j_pos == 0xFFFFFFFFu || t < j_t || (t == j_t && oid < j_oid))) {                     \
        j_t = t; j_pos = (position); j_oid = oid; j_u = u; j_v = v;                                    \
      }                                                                                                \
    }                                                                                                  \
  } while (0)
// Faces from..cnt - 1 of the leaf at position 'first'.
#define RK_LEAF_HITS(first, from, cnt)                                                                 \
  for (uint32_t k = (from); k < (cnt); ++k) {                                                          \
    const float4* tri_ = tris + 3 * (size_t)((first) + k);                                             \
    const float4 a_ = tri_[0], b_ = tri_[1], c_ = tri_[2];                                             \
    RK_TRI_HIT(a_, b_, c_, (first) + k);                                                               \
  }

//
// kBoundEvery: helpers read their owner's best so far on every kBoundEvery-th
// step only (1: every step); in between they cull against the value they last
// read, which can only be larger, so they may visit more nodes but find the
// same closest hit.
//
// kApart: leaves' triangles are loaded by instructions of their own, after the
// nodes' and before the one wait, for rays that share no nodes. With both in one
// instruction such rays fetch lines into the L1 more than once: 2M incoherent rays on
// 250,000 faces made 279M requests to the L2 and took 2.35 ms, apart 217M and 1.79.
template <bool kCount, int kStackN, int kLds, int kWG, bool kOldest = false, int kLeafBatch = 0,
          int kDonateMin = 1, int kBoundEvery = 1, bool kApart = false>
__device__ __forceinline__ RayHit trace_ray_shared(const FNode* __restrict__ nodes, const float4* __restrict__ tris,
                                                   uint32_t n_tris, uint32_t root, bool has_ray, float4 orig,
                                                   float4 dir, float depth0, float eps, uint32_t& n_box,
                                                   uint32_t& n_tri, uint2* lds, uint32_t* xchg) {
  const uint32_t lane = __lane_id();
  const uint32_t max_visits = 4 * n_tris + 64;  // a subtree visit touches each node once
  // this lane's own ray: its best hit
  uint32_t o_pos = 0xFFFFFFFFu, o_oid = 0xFFFFFFFFu;
  float o_t = depth0, o_u = 0.0f, o_v = 0.0f;
  // the job: a subtree (cur + stack) of the owner's ray, and a helper's own best
  int owner = has_ray ? (int)lane : -1;
  float4 jo = orig, jd = dir;
  float ix = safe_inv(jd.x), iy = safe_inv(jd.y), iz = safe_inv(jd.z);
  float ox = jo.x * ix, oy = jo.y * iy, oz = jo.z * iz;
  uint32_t j_pos = 0xFFFFFFFFu, j_oid = 0xFFFFFFFFu;
  float j_t = RK_HUGE, j_u = 0.0f, j_v = 0.0f;
  uint32_t cur = root, visits = 0;
  uint32_t pend = 0u;  // a postponed leaf (a leaf reference always has kLeafBit set; 0: none)
  uint32_t step = 0;   // loop steps so far (the same in every lane)
  float h_t = depth0;  // kBoundEvery > 1: the owner's best as this helper last read it
  bool h_hit = false;
  static_assert(kStackN > kLds, "scratch part of the stack");
  uint32_t stack_ref[kStackN - kLds];
  float stack_t[kStackN - kLds];
  // An LDS-typed pointer (an entry is ref | t << 32, the layout of a uint2):
  // with a generic one the compiler merges the two branches of st_get into one
  // flat load through a selected address, which costs a flat access (and a
  // wait on every memory counter) per pop.
  typedef __attribute__((address_space(3))) unsigned long long lds_u64;
  lds_u64* my_lds = (lds_u64*)(lds + threadIdx.x);
  int sp = 0, sb = 0;
  auto st_get = [&](int i, uint32_t& r, float& t) {
    if (i < kLds) {
      const unsigned long long e = my_lds[i * kWG];
      r = (uint32_t)e;
      t = __uint_as_float((uint32_t)(e >> 32));
    } else {
      r = stack_ref[i - kLds];
      t = stack_t[i - kLds];
    }
  };
  auto st_set = [&](int i, uint32_t r, float t) {
    if (i < kLds) {
      my_lds[i * kWG] = (unsigned long long)r | ((unsigned long long)__float_as_uint(t) << 32);
    } else {
      stack_ref[i - kLds] = r;
      stack_t[i - kLds] = t;
    }
  };
  for (;;) {
    const bool working = owner >= 0;
    const uint64_t idle = __ballot(!working);
    if (idle == ~0ull) break;
    bool fresh = false;  // this lane took a new job this step
    // hand the newest pending subtree of up to popc(idle) lanes to idle lanes
    const uint64_t donors = __ballot(working && sp > sb);
    if (idle != 0ull && donors != 0ull && (kDonateMin <= 1 || __popcll(idle) >= kDonateMin)) {
      const uint32_t nd = min((uint32_t)__popcll(idle), (uint32_t)__popcll(donors));
      const uint64_t lt = rk::lanemask_lt();
      const uint32_t rd = (uint32_t)__popcll(donors & lt), ri = (uint32_t)__popcll(idle & lt);
      if (working && sp > sb && rd < nd) {
        // the newest entry: taking it is a pop, so the stack stays one
        // entry per level of the current path at most (kOldest: the oldest)
        uint32_t r0;
        float t0;
        if (kOldest) {
          st_get(sb, r0, t0);
          if (++sb == sp) sb = sp = 0;
        } else {
          --sp;
          st_get(sp, r0, t0);
        }
        __hip_atomic_store(xchg + rd, r0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        __hip_atomic_store(xchg + kXchg + rd, __float_as_uint(t0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        __hip_atomic_store(xchg + 2 * kXchg + rd, (uint32_t)owner, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        __hip_atomic_store(xchg + 3 * kXchg + rd, lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
      __builtin_amdgcn_wave_barrier();
      const bool take = !working && ri < nd;
      uint32_t g_ref = 0, g_t = 0, g_own = lane, g_don = lane;
      if (take) {
        g_ref = __hip_atomic_load(xchg + ri, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        g_t = __hip_atomic_load(xchg + kXchg + ri, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        g_own = __hip_atomic_load(xchg + 2 * kXchg + ri, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        g_don = __hip_atomic_load(xchg + 3 * kXchg + ri, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
      __builtin_amdgcn_wave_barrier();
      // Every lane takes part in the exchange. The donor's job is a subtree of
      // the owner's ray, so the donor holds that ray and its slab terms (the
      // same bits the owner computed): copying them saves three divisions.
      const int src = (int)g_own, don = (int)g_don;
      const float4 no = make_float4(__shfl(jo.x, don, 64), __shfl(jo.y, don, 64), __shfl(jo.z, don, 64),
                                    __shfl(jo.w, don, 64));
      const float4 ndr = make_float4(__shfl(jd.x, don, 64), __shfl(jd.y, don, 64), __shfl(jd.z, don, 64),
                                     __shfl(jd.w, don, 64));
      const float nix = __shfl(ix, don, 64), niy = __shfl(iy, don, 64), niz = __shfl(iz, don, 64);
      const float nox = __shfl(ox, don, 64), noy = __shfl(oy, don, 64), noz = __shfl(oz, don, 64);
      const float od = __shfl(o_t, src, 64);
      if (take && __uint_as_float(g_t) <= od) {
        fresh = true;
        owner = src;
        jo = no;
        jd = ndr;
        ix = nix;
        iy = niy;
        iz = niz;
        ox = nox;
        oy = noy;
        oz = noz;
        cur = g_ref;
        sp = 0;
        sb = 0;
        visits = 0;
        j_pos = 0xFFFFFFFFu;
        j_t = RK_HUGE;
        j_oid = 0xFFFFFFFFu;
      }
    }
    const bool own = owner == (int)lane;
    // This step's record, a node or a leaf's first triangle, is fetched here for
    // both kinds of lanes, with one wait where there would be one in each branch,
    // and meanwhile the owner's bound is read; its address is computed without a
    // branch. It takes 80 registers, not 64, and 24 waves per CU that wait once are
    // faster than 32 that wait twice: the 1024-mesh batch 4.35 -> 3.95 ms, the 1920x1080
    // heightfield frame 192 -> 167 us (179 with branches for the address, and then the
    // 1380x1035 frame of a small heightfield 82 -> 90), the
    // 256x256 icosphere frame 63 -> 55, 32 served requests 3.50 -> 3.03 ms.
    const bool at_leaf = (cur & kLeafBit) != 0u;
    const uint32_t first = (cur & ~kLeafBit) >> 4;
    const uint32_t idx = at_leaf ? first : cur;
    const bool in_tree = idx < n_tris;
    float4 q0, q1, q2;
    float2 q3;
    if (owner >= 0 && in_tree && !(at_leaf && (kLeafBatch != 0 || kApart))) {
      const uint64_t base = at_leaf ? reinterpret_cast<uint64_t>(tris) : reinterpret_cast<uint64_t>(nodes);
      const float4* rec = reinterpret_cast<const float4*>(base + (uint64_t)idx * (at_leaf ? 48u : 64u));
      q0 = rec[0];
      q1 = rec[1];
      q2 = rec[2];
      if (!at_leaf) q3 = *reinterpret_cast<const float2*>(rec + 3);
    }
    if (kApart && kLeafBatch == 0 && owner >= 0 && in_tree && at_leaf) {
      const float4* rec = tris + 3 * (size_t)idx;
      q0 = rec[0];
      q1 = rec[1];
      q2 = rec[2];
    }
    // the owner's best so far bounds a helper's subtree
    float dmax = o_t;
    bool d_hit = o_pos != 0xFFFFFFFFu;
    // a lane that just took a job reads its new owner's bound at once
    if (kBoundEvery <= 1 || (step % (uint32_t)kBoundEvery) == 0u || __ballot(fresh) != 0ull) {
      if (__ballot(owner >= 0 && !own) != 0ull) {
        const int src = owner >= 0 ? owner : (int)lane;
        const float od = __shfl(o_t, src, 64);
        const uint32_t op = __shfl(o_pos, src, 64);
        if (!own) {
          dmax = od;
          d_hit = op != 0xFFFFFFFFu;
        }
      }
      if (kBoundEvery > 1) {
        h_t = dmax;
        h_hit = d_hit;
      }
    } else if (!own) {
      dmax = h_t;
      d_hit = h_hit;
    }
    ++step;
    bool job_end = false, flush_me = false, end_after = false;
    if (owner >= 0) {
      // an owner's dmax is its o_t; its j_t, and a helper's without a hit, are RK_HUGE
      float bound = j_t < dmax ? j_t : dmax;
      bool need_pop = false;
      if (++visits > max_visits || !(in_tree || at_leaf)) {
        job_end = true;  // never taken for a tree built here
        pend = 0u;
      } else if (!at_leaf) {
        FNode nd;
        nd.a = q0;
        nd.b = q1;
        nd.c = q2;
        nd.d = make_uint4(__float_as_uint(q3.x), __float_as_uint(q3.y), 0u, 0u);
        const Slab2 sl = slab2(nd, ix, iy, iz, ox, oy, oz, bound);
        const float tmin0 = sl.tmin0, tmin1 = sl.tmin1;
        const bool h0 = sl.h0, h1 = sl.h1;
        if (kCount) n_box += 2;
        if (h0 && h1) {
          const bool first0 = tmin0 <= tmin1;
          if (sp < kStackN) {
            st_set(sp, first0 ? nd.d.y : nd.d.x, first0 ? tmin1 : tmin0);
            ++sp;
          }
          cur = first0 ? nd.d.x : nd.d.y;
        } else if (h0) {
          cur = nd.d.x;
        } else if (h1) {
          cur = nd.d.y;
        } else {
          need_pop = true;
        }
      } else if (kLeafBatch == 0) {
        if (in_tree) {
          RK_TRI_HIT(q0, q1, q2, first);
          if ((cur & 15u) != 0u) {
            const uint32_t cnt = min((cur & 15u) + 1u, n_tris - first);
            RK_LEAF_HITS(first, 1u, cnt);
          }
        }
        need_pop = true;
      } else if (pend == 0u) {
        pend = cur;  // postponed: go on to the next pending subtree
        need_pop = true;
      } else {
        flush_me = true;  // a second leaf: test the pending one first, keep cur
      }
      if (need_pop) {
        // the nearest pending entry that can still hold a closer hit
        const float lim = own ? o_t : dmax;
        bound = j_t < lim ? j_t : lim;
        bool found = false;
        while (sp > sb) {
          --sp;
          uint32_t r;
          float t;
          st_get(sp, r, t);
          if (t <= bound) {
            cur = r;
            found = true;
            break;
          }
        }
        if (!found) {
          if (kLeafBatch > 0 && pend != 0u) {
            flush_me = true;  // the subtree is done but for its pending leaf
            end_after = true;
          } else {
            job_end = true;
          }
        }
      }
    }
    if (kLeafBatch > 0) {
      const uint64_t pm = __ballot(pend != 0u);
      if (pm != 0ull && (__ballot(flush_me) != 0ull || __popcll(pm) >= kLeafBatch)) {
        if (pend != 0u) {
          const uint32_t p_first = (pend & ~kLeafBit) >> 4;
          const uint32_t p_cnt = p_first < n_tris ? min((pend & 15u) + 1u, n_tris - p_first) : 0u;
          RK_LEAF_HITS(p_first, 0u, p_cnt);
          pend = 0u;
        }
        if (end_after) job_end = true;
      }
    }
    // merge finished helpers' hits into their owners, one at a time
    uint64_t m = __ballot(job_end && !own && j_pos != 0xFFFFFFFFu);
    while (m != 0ull) {
      const int e = __builtin_ctzll(m);
      m &= m - 1;
      const int ow = __shfl(owner, e, 64);
      const float ct = __shfl(j_t, e, 64);
      const uint32_t coid = __shfl(j_oid, e, 64), cpos = __shfl(j_pos, e, 64);
      const float cu = __shfl(j_u, e, 64), cv = __shfl(j_v, e, 64);
      if ((int)lane == ow && (ct < o_t || (o_pos != 0xFFFFFFFFu && ct == o_t && coid < o_oid))) {
        o_t = ct; o_pos = cpos; o_oid = coid; o_u = cu; o_v = cv;
      }
    }
    if (job_end) owner = -1;
  }
  return RayHit{o_pos, o_t, o_u, o_v};
}
#undef RK_LEAF_HITS
#undef RK_TRI_HIT

// Sort key of a ray: the 30-bit Morton code of its origin in the tree's root
// box (the union of the root record's two child boxes), clamped to the box.
__global__ __launch_bounds__(256) void k_ray_keys(const FNode* __restrict__ nodes, const float4* __restrict__ origins,
                                                  uint32_t n, uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ vals) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const FNode r = nodes[0];
  const float lx = rk::fmn(r.a.x, r.b.x), hx = rk::fmx(r.a.y, r.b.y);
  const float ly = rk::fmn(r.a.z, r.b.z), hy = rk::fmx(r.a.w, r.b.w);
  const float lz = rk::fmn(r.c.x, r.c.z), hz = rk::fmx(r.c.y, r.c.w);
  const float4 o = origins[i];
  const uint32_t qx = min(rk::f2u_sat((o.x - lx) * (1024.0f / (hx - lx))), 1023u);
  const uint32_t qy = min(rk::f2u_sat((o.y - ly) * (1024.0f / (hy - ly))), 1023u);
  const uint32_t qz = min(rk::f2u_sat((o.z - lz) * (1024.0f / (hz - lz))), 1023u);
  keys[i] = (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz);
  vals[i] = i;
}

// Rays of one frame differ in cost by orders of magnitude: on a terrain seen
// at a low angle, the rays that graze the horizon make hundreds of node
// visits and the rays that leave the root box make one, and the grazing rays
// fill a few rows. A wave lasts as long as its costliest rays; its idle lanes
// help (trace_ray_shared), but a wave of 64 grazing rays has none idle. So a
// wave does not take 64 consecutive rays: it takes runs of kSpreadRun
// consecutive rays (a 128-B line of origins and one of directions) from
// 64 / kSpreadRun bands of the ray array, the run at the same place in each
// band. Runs of 8 measured best on the 1920x1080 heightfield frame (with help at
// one idle lane 0.176 ms against 0.283 for 64 consecutive rays; 0.219 for runs of
// 4, 0.200 for runs of 16). 0 traces the rays in array order. Sorted traces keep
// their order.
#ifndef RK_TRACE_SPREAD
#define RK_TRACE_SPREAD 8
#endif
constexpr uint32_t kSpreadRun = RK_TRACE_SPREAD;

// The ray of thread t (n_rays when none).
__device__ __forceinline__ uint32_t spread_ray(uint32_t t, uint32_t n_rays) {
  return rk::band_ray<kSpreadRun>(t, n_rays);
}

// order (may be NULL): thread t traces ray order[t], so rays that start near
// each other run in the same wave; results still go to the ray's own slot.
// Threads per workgroup of k_fast_trace and k_fast_trace_camera. One wave per
// workgroup: a finished wave frees its slot at once, where a larger workgroup
// waits for its slowest wave. On the 1920x1080 heightfield frame 64, 128 and 256
// threads take 0.176, 0.175 and 0.181 ms (camera 0.173 and 0.171) with help at one
// idle lane, and are within 1% on the 10M soup's incoherent rays. (Before a step
// fetched in one place 64 was ahead: 0.211, 0.218, 0.228 ms.)
#ifndef RK_TRACE_WG
#define RK_TRACE_WG 64
#endif
constexpr int kTraceWG = RK_TRACE_WG;
// Pending subtrees are handed to idle lanes only on steps where at least this
// many lanes are idle (trace_ray_shared's kDonateMin): each exchange costs
// every lane of the wave a dozen shuffles and two LDS round trips, and a lane
// that waits a few steps for work costs less. 16 measured best on the
// 1920x1080 heightfield frame (0.166 ms against 0.177 with 1, 0.171 with 8 and
// 0.190 with 32); trees past the L2 take 32 (kFetchBoundFaces, kMemoryFaces).
#ifndef RK_TRACE_DONATE_MIN
#define RK_TRACE_DONATE_MIN 16
#endif
constexpr int kTraceDonateMin = RK_TRACE_DONATE_MIN;
static_assert(kTraceWG % 64 == 0 && kTraceWG <= 1024, "whole waves");

// Sorted rays of a tree that the eight L2s cannot hold between them: workgroups are
// dealt to the XCDs in turn, so consecutive ones would fetch the same nodes into all
// eight L2s. With kXcdRuns an XCD takes runs of kXcdRun consecutive workgroups of the
// order, on trees of kXcdFaces on. Sort and trace of 300k, 1M and 4M rays: on 600k faces
// 570 -> 512, 1,280 -> 1,225 and 4,300 -> 4,300 us, on 10M faces 957 -> 871, 2,330 -> 2,075
// and 7,250 -> 6,230; 16M on 10M 24.6 -> 23.9 ms. 2M on 300k faces, 1.71 -> 1.78, are the
// one slower. Runs of 32, 128 and 512 are within 4%.
constexpr uint32_t kXcdRun = 512, kXcdFaces = 1u << 18;
// And from this many faces on, where what bounds the trace is fetching nodes past
// the L2, idle lanes take subtrees (which the owner might have culled) only on steps
// where half the wave is idle: 16M rays on the 10M soup 26.8 -> 23.9 ms, 8M on 3M
// faces 13.5 -> 12.4, 4M on 1M 5.17 -> 4.97. On fewer faces it depends on the rays: 300k and
// 4M on 400k faces 438 -> 476 us and 3.69 -> 3.62 ms.
constexpr uint32_t kFetchBoundFaces = 1u << 20;
// Rays in array order may be a picture's, whose rays share nodes and gain from early
// help, so the same holds only from where the tree is beyond the 256 MB memory-side cache
// too: 16M rays on the 10M soup 45.0 -> 38.7 ms; a 1920x1080 frame of a 3.9M-face heightfield
// would go from 234 us to 289, as long as it took before nodes and leaves were
// fetched together.
constexpr uint32_t kMemoryFaces = 1u << 22;

// Sorted rays fetch leaves apart (kApart) from this many faces on. Which is better
// depends on how much the rays hit. Sort and trace of 4M rays on soups of the same area
// (about one hit in two), 20,000, 80,000, 150,000, 500,000 and 1M faces: together 2.12, 2.29,
// 2.44, 2.98 and 3.64 ms, apart 2.25, 2.42, 2.53, 2.93 and 3.36. 2M rays on 70,000, 150,000 and
// 300,000 small faces, of which few are hit: 1.10, 1.61 and 2.28 ms, apart 0.95, 1.29 and
// 1.78. In array order all fetch together: pictures, which gain 2-30% from it, cannot
// be told from rays that share no nodes (those lose up to 25% on 50,000 to 1M small
// faces) but by a test of the waves' origins, which costs pictures 0.5-2%, and with both
// loops in a kernel 3 registers spill, which costs rays that hit much 15%.
constexpr uint32_t kApartFaces = 1u << 17;

// kWG threads per workgroup, runs of kRun rays per band (spread_ray; 0: 64
// consecutive rays per wave), kLds stack entries per lane in LDS. The
// defaults above are one variant; rk_fast_autotune chooses among several.
template <bool kCount, int kWG, uint32_t kRun, int kLds, bool kOldest = false, int kLeafBatch = 0, int kDonateMin = 1,
          int kBoundEvery = 1, bool kXcdRuns = false, bool kApart = false>
__global__ __launch_bounds__(kWG) void k_fast_trace_v(const FNode* __restrict__ nodes, const float4* __restrict__ tris,
                                                      uint32_t n_tris, const float4* __restrict__ origins,
                                                      const float4* __restrict__ dirs, uint32_t n_rays,
                                                      uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                      float* __restrict__ depths, float eps,
                                                      unsigned long long* __restrict__ counters,
                                                      const uint32_t* __restrict__ order, uint32_t flags) {
  uint32_t block = blockIdx.x;
  if (kXcdRuns) {
    const uint32_t group = block / (8u * kXcdRun) * (8u * kXcdRun), i = block - group;
    if (group + 8u * kXcdRun <= gridDim.x) block = group + (i & 7u) * kXcdRun + (i >> 3);
  }
  const uint32_t t = block * kWG + threadIdx.x;
  const bool reset = (flags & RK_TRACE_RESET_DEPTH) != 0u;
  const uint32_t l = order ? (t < n_rays ? order[t] : n_rays) : rk::band_ray<kRun>(t, n_rays);
  const bool has_ray = l < n_rays;
  __shared__ uint2 s_stack[kLds * kWG];
  __shared__ uint32_t s_xchg[kWG / 64][kXchgWords];
  uint32_t n_box = 0, n_tri = 0;
  const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const RayHit h = trace_ray_shared<kCount, kStack, kLds, kWG, kOldest, kLeafBatch, kDonateMin, kBoundEvery, kApart>(
      nodes, tris, n_tris, 0u, has_ray, has_ray ? origins[l] : zero4, has_ray ? dirs[l] : zero4,
      has_ray ? (reset ? RK_HUGE : depths[l]) : 0.0f, eps, n_box, n_tri, s_stack, s_xchg[threadIdx.x >> 6]);
  if (kCount) {
    atomicAdd(counters, (unsigned long long)n_box);
    atomicAdd(counters + 1, (unsigned long long)n_tri);
  }
  if (has_ray) {
    if (h.pos != 0xFFFFFFFFu) {
      faces_id[l] = h.pos;
      coords[l] = make_float2(h.u, h.v);
      depths[l] = h.t;
    } else if (reset) {
      depths[l] = RK_HUGE;  // the reset a fill kernel would have done; the miss's id and coords stay
    }
  }
}

inline unsigned blocks_for(uint32_t n, uint32_t per) { return (n + per - 1) / per; }

// Workspace of the hierarchy passes over n positions. What callers know of it, its
// size, the no-allocation build's face limits and what is refused as too small, has
// two words per position that no pass uses: they are taken all the same.
struct HierWs {
  HierItem* items;   // the subtrees each chunk, then each group of chunks, left over
  uint32_t* counts;  // per chunk, how many
};
inline size_t hier_ws_bytes(size_t n) {
  return rk_align_up(n * 4) + rk_align_up(n * sizeof(HierItem)) + rk_align_up(n * 4) +
         rk_align_up(((n + kChunk - 1) / kChunk) * 4);
}
inline bool take_hier_ws(RkArena& ar, uint32_t n, HierWs& w) {
  const bool first = ar.take<uint32_t>(n) != nullptr;
  w.items = ar.take<HierItem>(n);
  const bool second = ar.take<uint32_t>(n) != nullptr;
  w.counts = ar.take<uint32_t>((n + kChunk - 1) / kChunk);
  return first && w.items && second && w.counts;
}
// The chunk pass, then reductions of kReduceFan groups to one until one is left.
template <typename K, bool kBatch>
rk_status launch_hierarchy(hipStream_t st, const K* keys, const uint32_t* order, const uint4* f, const float4* v,
                           uint32_t n, uint32_t leaf_max, const HierWs& w, FNode* nodes, float4* tris,
                           const rk_batch_mesh* meshes) {
  const uint32_t chunks = blocks_for(n, kChunk);
  hipLaunchKernelGGL((k_fast_hierarchy<K, kBatch>), dim3(chunks), dim3(kChunk), 0, st, keys, order, f, v, n, leaf_max,
                     nodes, tris, meshes, w.items, w.counts);
  RK_CHECK_LAUNCH();
  uint32_t stride = 1;
  for (uint32_t groups = chunks; groups > 1; stride *= kReduceFan) {
    const bool small = groups <= (stride == 1 ? kReduceSmall : kReduceSmallGroups);
    groups = blocks_for(groups, kReduceFan);
    if (small)
      hipLaunchKernelGGL((k_hier_reduce<K, kBatch, 512>), dim3(groups), dim3(512), 0, st, keys, n, leaf_max, chunks,
                         stride, nodes, w.items, w.counts);
    else
      hipLaunchKernelGGL((k_hier_reduce<K, kBatch, 1024>), dim3(groups), dim3(1024), 0, st, keys, n, leaf_max, chunks,
                         stride, nodes, w.items, w.counts);
    RK_CHECK_LAUNCH();
  }
  return RK_SUCCESS;
}

}  // namespace

extern "C" size_t rk_fast_build_workspace_size(uint32_t face_count, int morton_mode) {
  size_t n = face_count ? face_count : 1;
  size_t kb = morton_mode == RK_MORTON_63 ? 8 : 4;
  size_t b = 0;
  b += rk_align_up(n * kb);               // keys
  b += hier_ws_bytes(n);
  b += rk_sort_workspace_size((uint32_t)n, (uint32_t)kb);
  return b + 4096;
}

template <typename K>
static rk_status fast_build_keys(hipStream_t st, const uint4* f, const float4* v, uint32_t n, float4 rmin,
                                 float4 rmax, const rk_fast_bvh* bvh, uint32_t leaf_max, K* keys, const HierWs& hw,
                                 void* sort_ws, size_t sort_bytes, uint32_t* info) {
  constexpr int kKeyBits = sizeof(K) == 4 ? 30 : 63;
  uint32_t* order = bvh->indices;
  RkSortPlan<K> plan;
  rk_status s = rk_sort_plan<K>(n, kKeyBits, true, keys, order, sort_ws, sort_bytes, plan);
  if (s != RK_SUCCESS) return s;
  // Below 2^21 faces the key kernel counts the sort's digits as well (1M
  // faces: 14.4 us, and 4.9 to clear the counts, against 15.5 and 13.2 for a
  // kernel of its own); above, its LDS atomics cost what that kernel does
  // (10M faces, 63-bit keys: 274 against 203 + 65 us).
  const bool counted = !plan.one && n < kCountInPrep;
  if (counted && (s = rk_sort_clear<K>(st, plan, info)) != RK_SUCCESS) return s;
  const uint32_t per = counted && n >= kCountPer4 ? 4u : 1u;
  auto prep = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks_for(n, per * kPrepThreads)), dim3(kPrepThreads), 0, st, f, v, n, rmin,
                       rmax, reinterpret_cast<Box*>(bvh->boxes), plan.src, plan.vsrc, info, per, plan.head + 1,
                       plan.copies);
  };
  if (counted) prep(k_fast_prep<K, (int)sizeof(K)>);
  else prep(k_fast_prep<K, 0>);
  RK_CHECK_LAUNCH();
  s = rk_sort_run<K>(st, plan, counted, info + RK_INFO_FLAGS);
  if (s != RK_SUCCESS) return s;
  return launch_hierarchy<K, false>(st, keys, order, f, v, n, leaf_max, hw, static_cast<FNode*>(bvh->nodes),
                                    static_cast<float4*>(bvh->tris), (const rk_batch_mesh*)nullptr);
}

static rk_status fast_build_common(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                   uint32_t face_count, const rk_aabox* hitbox, int morton_mode, uint32_t leaf_max,
                                   const rk_fast_bvh* bvh, uint32_t* info, void* sorted_keys, void* ws,
                                   size_t ws_bytes) {
  const uint32_t n = face_count;
  if (n == 0 || !faces || !vertices || !hitbox || !bvh || !info) return RK_ERROR_INVALID_VALUE;
  if (!bvh->nodes || !bvh->tris || !bvh->indices) return RK_ERROR_INVALID_VALUE;
  if (morton_mode != RK_MORTON_30 && morton_mode != RK_MORTON_63) return RK_ERROR_INVALID_VALUE;
  if (leaf_max < 1 || leaf_max > kMaxLeaf) return RK_ERROR_INVALID_VALUE;
  if (n >= (1u << 27)) return RK_ERROR_UNSUPPORTED;
  hipStream_t st = rk_hip_stream(stream);
  const bool wide = morton_mode == RK_MORTON_63;
  RkArena ar(ws, ws_bytes);
  void* keys = wide ? (void*)ar.take<uint64_t>(n) : (void*)ar.take<uint32_t>(n);
  HierWs hw;
  const bool hw_ok = take_hier_ws(ar, n, hw);
  const size_t sort_bytes = rk_sort_workspace_size(n, wide ? 8 : 4);
  void* sort_ws = ar.take<char>(sort_bytes);
  if (!keys || !hw_ok || !sort_ws) return RK_ERROR_WORKSPACE;
  if (sorted_keys) keys = sorted_keys;
  float4 rmin = make_float4(hitbox->min.x, hitbox->min.y, hitbox->min.z, hitbox->min.w);
  float4 rmax = make_float4(hitbox->max.x, hitbox->max.y, hitbox->max.z, hitbox->max.w);
  const uint4* f = reinterpret_cast<const uint4*>(faces);
  const float4* v = reinterpret_cast<const float4*>(vertices);
  if (wide)
    return fast_build_keys<uint64_t>(st, f, v, n, rmin, rmax, bvh, leaf_max, static_cast<uint64_t*>(keys), hw,
                                     sort_ws, sort_bytes, info);
  return fast_build_keys<uint32_t>(st, f, v, n, rmin, rmax, bvh, leaf_max, static_cast<uint32_t*>(keys), hw,
                                   sort_ws, sort_bytes, info);
}

extern "C" rk_status rk_fast_build(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                   uint32_t face_count, const rk_aabox* hitbox, int morton_mode, uint32_t leaf_max,
                                   const rk_fast_bvh* bvh, uint32_t* info, void* ws, size_t ws_bytes) {
  return fast_build_common(stream, faces, vertices, face_count, hitbox, morton_mode, leaf_max, bvh, info, nullptr,
                           ws, ws_bytes);
}

extern "C" rk_status rk_fast_build_keyed(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                         uint32_t face_count, const rk_aabox* hitbox, int morton_mode,
                                         uint32_t leaf_max, const rk_fast_bvh* bvh, uint32_t* info, void* sorted_keys,
                                         void* ws, size_t ws_bytes) {
  if (!sorted_keys) return RK_ERROR_INVALID_VALUE;
  return fast_build_common(stream, faces, vertices, face_count, hitbox, morton_mode, leaf_max, bvh, info,
                           sorted_keys, ws, ws_bytes);
}

// ---- rk_fast_build without a caller workspace ------------------------------------
// The workspace of rk_fast_build (keys, hierarchy slots and counters, sort
// buffers and look-back status) lives in one file-scope device array. Every
// device the library runs on holds its own copy until the process ends. Host
// code never passes the array's name to a kernel: the device address comes
// from hipGetSymbolAddress, once per device, on that device's first call.
namespace {
constexpr size_t kNoAllocScratchBytes = RK_NOALLOC_SCRATCH_BYTES;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

rk_status scratch_for_current_device(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return RK_ERROR_DEVICE;
  if (dev < 0 || dev >= kMaxDevices) return RK_ERROR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return RK_ERROR_DEVICE;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return RK_SUCCESS;
}
}  // namespace

extern "C" rk_status rk_fast_build_noalloc(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                           uint32_t face_count, const rk_aabox* hitbox, int morton_mode,
                                           uint32_t leaf_max, const rk_fast_bvh* bvh, uint32_t* info) {
  if (morton_mode != RK_MORTON_30 && morton_mode != RK_MORTON_63) return RK_ERROR_INVALID_VALUE;
  if (face_count >= (1u << 27) || rk_fast_build_workspace_size(face_count, morton_mode) > kNoAllocScratchBytes)
    return RK_ERROR_WORKSPACE;
  void* ws = nullptr;
  rk_status s = scratch_for_current_device(&ws);
  if (s != RK_SUCCESS) return s;
  return fast_build_common(stream, faces, vertices, face_count, hitbox, morton_mode, leaf_max, bvh, info, nullptr, ws,
                           kNoAllocScratchBytes);
}

extern "C" rk_status rk_fast_refit(rk_stream stream, const rk_uint4* faces, const rk_float4* vertices,
                                   uint32_t face_count, int morton_mode, uint32_t leaf_max, const rk_fast_bvh* bvh,
                                   const void* sorted_keys, void* ws, size_t ws_bytes) {
  const uint32_t n = face_count;
  if (n == 0 || !faces || !vertices || !bvh || !sorted_keys) return RK_ERROR_INVALID_VALUE;
  if (!bvh->nodes || !bvh->tris || !bvh->indices) return RK_ERROR_INVALID_VALUE;
  if (morton_mode != RK_MORTON_30 && morton_mode != RK_MORTON_63) return RK_ERROR_INVALID_VALUE;
  if (leaf_max < 1 || leaf_max > kMaxLeaf) return RK_ERROR_INVALID_VALUE;
  if (n >= (1u << 27)) return RK_ERROR_UNSUPPORTED;
  hipStream_t st = rk_hip_stream(stream);
  RkArena ar(ws, ws_bytes);
  HierWs hw;
  if (!take_hier_ws(ar, n, hw)) return RK_ERROR_WORKSPACE;
  const uint4* f = reinterpret_cast<const uint4*>(faces);
  const float4* v = reinterpret_cast<const float4*>(vertices);
  FNode* nodes = static_cast<FNode*>(bvh->nodes);
  float4* tris = static_cast<float4*>(bvh->tris);
  if (morton_mode == RK_MORTON_63)
    return launch_hierarchy<uint64_t, false>(st, static_cast<const uint64_t*>(sorted_keys), bvh->indices, f, v, n,
                                             leaf_max, hw, nodes, tris, (const rk_batch_mesh*)nullptr);
  return launch_hierarchy<uint32_t, false>(st, static_cast<const uint32_t*>(sorted_keys), bvh->indices, f, v, n,
                                           leaf_max, hw, nodes, tris, (const rk_batch_mesh*)nullptr);
}


// ---- batches ------------------------------------------------------------------

namespace {

// The mesh whose [offset, offset + count) holds g, for offsets in increasing
// order (mesh_count >= 1): the last mesh with offset <= g.
__device__ __forceinline__ uint32_t mesh_of_face(const rk_batch_mesh* __restrict__ meshes, uint32_t mesh_count,
                                                 uint32_t g) {
  uint32_t lo = 0, hi = mesh_count - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (meshes[mid].face_offset <= g) lo = mid; else hi = mid - 1;
  }
  return lo;
}
__device__ __forceinline__ uint32_t mesh_of_ray(const rk_batch_mesh* __restrict__ meshes, uint32_t mesh_count,
                                                uint32_t r) {
  uint32_t lo = 0, hi = mesh_count - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (meshes[mid].ray_offset <= r) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Per-face box centroid quantised to 10 bits per axis in its mesh's hitbox,
// keyed (mesh << 30 | code) so one sort orders every mesh at once.
__global__ __launch_bounds__(256) void k_batch_prep(const rk_batch_mesh* __restrict__ meshes, uint32_t mesh_count,
                                                    const uint4* __restrict__ faces, const float4* __restrict__ verts,
                                                    uint32_t n, const rk_aabox* __restrict__ hitboxes,
                                                    uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t g = blockIdx.x * 256 + threadIdx.x;
  if (g >= n) return;
  const uint32_t m = mesh_of_face(meshes, mesh_count, g);
  const uint32_t voff = meshes[m].vertex_offset;
  const uint4 f = faces[g];
  const float4 v0 = verts[f.x + voff], v1 = verts[f.y + voff], v2 = verts[f.z + voff];
  const float4 mn = rk::min4(rk::min4(v0, v1), v2), mx = rk::max4(rk::max4(v0, v1), v2);
  const rk_aabox hb = hitboxes[m];
  const float4 rmin = make_float4(hb.min.x, hb.min.y, hb.min.z, 0.0f);
  const float4 len = make_float4(hb.max.x - hb.min.x, hb.max.y - hb.min.y, hb.max.z - hb.min.z, 0.0f);
  const float4 c = rk::muls4(rk::add4(mn, mx), 0.5f);
  const float sx = 1024.0f / len.x, sy = 1024.0f / len.y, sz = 1024.0f / len.z;
  const uint32_t qx = min(rk::f2u_sat((c.x - rmin.x) * sx), 1023u);
  const uint32_t qy = min(rk::f2u_sat((c.y - rmin.y) * sy), 1023u);
  const uint32_t qz = min(rk::f2u_sat((c.z - rmin.z) * sz), 1023u);
  keys[g] = ((uint64_t)m << 30) | (uint64_t)((spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz));
  vals[g] = g;
}

// Sort key of ray r: (mesh << 30 | 30-bit Morton code of its origin in the
// mesh's root box), so one sort orders the rays of every mesh by where they
// start and keeps each mesh's rays together. A mesh of one face has no root
// record and keys all its rays alike.
__global__ __launch_bounds__(256) void k_batch_ray_keys(const rk_batch_mesh* __restrict__ meshes,
                                                        uint32_t mesh_count, const FNode* __restrict__ nodes,
                                                        const float4* __restrict__ origins, uint32_t n,
                                                        uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t r = blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  const uint32_t m = mesh_of_ray(meshes, mesh_count, r);
  uint32_t code = 0;
  if (meshes[m].face_count >= 2) {
    const FNode root = nodes[meshes[m].face_offset];
    const float lx = rk::fmn(root.a.x, root.b.x), hx = rk::fmx(root.a.y, root.b.y);
    const float ly = rk::fmn(root.a.z, root.b.z), hy = rk::fmx(root.a.w, root.b.w);
    const float lz = rk::fmn(root.c.x, root.c.z), hz = rk::fmx(root.c.y, root.c.w);
    const float4 o = origins[r];
    const uint32_t qx = min(rk::f2u_sat((o.x - lx) * (1024.0f / (hx - lx))), 1023u);
    const uint32_t qy = min(rk::f2u_sat((o.y - ly) * (1024.0f / (hy - ly))), 1023u);
    const uint32_t qz = min(rk::f2u_sat((o.z - lz) * (1024.0f / (hz - lz))), 1023u);
    code = (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz);
  }
  keys[r] = ((uint64_t)m << 30) | code;
  vals[r] = r;
}

// Closest hit of ray r (r >= n_rays: none, the lane only helps the others of
// its wave), in its mesh's tree. Every lane of the wave calls it.
template <int kStackN, int kWG, int kDM>
__device__ __forceinline__ void batch_trace_one(const rk_batch_mesh* __restrict__ meshes, uint32_t mesh_count,
                                                const FNode* __restrict__ nodes, const float4* __restrict__ tris,
                                                uint32_t n_tris, const float4* __restrict__ origins,
                                                const float4* __restrict__ dirs, uint32_t r, uint32_t n_rays,
                                                uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                float* __restrict__ depths, float eps, uint2* lds_stack,
                                                uint32_t* xchg) {
  const bool has_ray = r < n_rays;
  const uint32_t root = has_ray ? meshes[mesh_of_ray(meshes, mesh_count, r)].face_offset : 0u;
  const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  uint32_t nb = 0, nt = 0;
  const RayHit h = trace_ray_shared<false, kStackN, kDeepLdsStack, kWG, false, 0, kDM>(
      nodes, tris, n_tris, root, has_ray, has_ray ? origins[r] : zero4, has_ray ? dirs[r] : zero4,
      has_ray ? depths[r] : 0.0f, eps, nb, nt, lds_stack, xchg);
  if (has_ray && h.pos != 0xFFFFFFFFu) {
    faces_id[r] = h.pos;
    coords[r] = make_float2(h.u, h.v);
    depths[r] = h.t;
  }
}

// One ray per thread, kWG rays per workgroup.
template <int kWG, int kStackN, int kDM>
__global__ __launch_bounds__(kWG) void k_batch_trace_grid(const rk_batch_mesh* __restrict__ meshes,
                                                          uint32_t mesh_count, const FNode* __restrict__ nodes,
                                                          const float4* __restrict__ tris, uint32_t n_tris,
                                                          const float4* __restrict__ origins,
                                                          const float4* __restrict__ dirs, uint32_t n_rays,
                                                          uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                          float* __restrict__ depths, float eps,
                                                          const uint32_t* __restrict__ order) {
  const uint32_t t = blockIdx.x * kWG + threadIdx.x;
  const uint32_t r = t < n_rays ? (order ? order[t] : t) : n_rays;
  __shared__ uint2 s_stack[kDeepLdsStack * kWG];
  __shared__ uint32_t s_xchg[kWG / 64][kXchgWords];
  batch_trace_one<kStackN, kWG, kDM>(meshes, mesh_count, nodes, tris, n_tris, origins, dirs, r, n_rays, faces_id, coords,
                                depths, eps, s_stack, s_xchg[threadIdx.x >> 6]);
}

// Persistent grid: every wave takes 64-ray tiles from its XCD's queue
// (workgroups are dealt to the eight XCDs in turn, so blockIdx % 8 is the
// XCD) and moves to the next queue once one runs dry; a queue that ran dry
// stays dry, so after eight dry queues in a row the wave has seen all work.
constexpr uint32_t kQueues = 8, kQueueStride = 32;  // counters 128 B apart

template <int kWG, int kStackN, int kDM>
__global__ __launch_bounds__(kWG) void k_batch_trace_queue(const rk_batch_mesh* __restrict__ meshes,
                                                           uint32_t mesh_count, const FNode* __restrict__ nodes,
                                                           const float4* __restrict__ tris, uint32_t n_tris,
                                                           const float4* __restrict__ origins,
                                                           const float4* __restrict__ dirs, uint32_t n_rays,
                                                           uint32_t* __restrict__ faces_id,
                                                           float2* __restrict__ coords, float* __restrict__ depths,
                                                           float eps, uint32_t* __restrict__ queues,
                                                           const uint32_t* __restrict__ order) {
  __shared__ uint2 s_stack[kDeepLdsStack * kWG];
  __shared__ uint32_t s_xchg[kWG / 64][kXchgWords];
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t n_tiles = (n_rays + 63) / 64;
  const uint32_t per = (n_tiles + kQueues - 1) / kQueues;
  uint32_t q = blockIdx.x % kQueues;
  for (uint32_t dry = 0; dry < kQueues;) {
    uint32_t t = 0;
    if (lane == 0) t = atomicAdd(queues + q * kQueueStride, 1u);
    t = __shfl(t, 0, 64);
    const uint32_t tile = q * per + t;
    if (t >= per || tile >= n_tiles) {
      q = (q + 1) % kQueues;
      ++dry;
      continue;
    }
    const uint32_t p = tile * 64 + lane;
    const uint32_t r = p < n_rays ? (order ? order[p] : p) : n_rays;
    batch_trace_one<kStackN, kWG, kDM>(meshes, mesh_count, nodes, tris, n_tris, origins, dirs, r, n_rays, faces_id, coords,
                                  depths, eps, s_stack, s_xchg[threadIdx.x >> 6]);
  }
}

int key_bits_for(uint32_t mesh_count) {
  int bits = 30;
  while (bits < 64 && (1ull << (bits - 30)) < mesh_count) ++bits;
  return bits;
}

bool config_ok(const rk_batch_config* c) {
  return c && c->leaf_max >= 1 && c->leaf_max <= kMaxLeaf && c->trace_mode <= 1 &&
         (c->trace_wg == 64 || c->trace_wg == 128 || c->trace_wg == 256) &&
         (c->stack_depth == 64 || c->stack_depth == 96) && c->ray_order <= 1 &&
         (c->donate_min == 0 || c->donate_min == (uint32_t)kTraceDonateMin || c->donate_min == 32);
}

}  // namespace

extern "C" rk_batch_config rk_batch_config_default(void) {
  rk_batch_config c = {};
  c.leaf_max = 1;
  c.trace_mode = 1;
  c.trace_wg = 256;
  c.stack_depth = 64;
  return c;
}

extern "C" size_t rk_batch_build_workspace_size(uint32_t mesh_count, uint32_t face_count) {
  (void)mesh_count;
  size_t n = face_count ? face_count : 1;
  size_t b = 0;
  b += rk_align_up(n * 8);  // (mesh, code) keys
  b += hier_ws_bytes(n);
  b += rk_sort_workspace_size((uint32_t)n, 8);
  return b + 4096;
}

extern "C" rk_status rk_batch_build(rk_stream stream, const rk_batch_mesh* meshes, uint32_t mesh_count,
                                    const rk_uint4* faces, const rk_float4* vertices, uint32_t face_count,
                                    const rk_aabox* hitboxes, const rk_batch_config* config, const rk_fast_bvh* bvh,
                                    uint32_t* info, void* ws, size_t ws_bytes) {
  const uint32_t n = face_count;
  if (!meshes || mesh_count == 0 || mesh_count > RK_BATCH_MAX_MESHES || n == 0 || !faces || !vertices ||
      !hitboxes || !bvh || !info || !config_ok(config))
    return RK_ERROR_INVALID_VALUE;
  if (!bvh->nodes || !bvh->tris || !bvh->indices) return RK_ERROR_INVALID_VALUE;
  if (n >= (1u << 27) || n < mesh_count) return RK_ERROR_UNSUPPORTED;
  hipStream_t st = rk_hip_stream(stream);
  RkArena ar(ws, ws_bytes);
  uint64_t* keys = ar.take<uint64_t>(n);
  HierWs hw;
  const bool hw_ok = take_hier_ws(ar, n, hw);
  const size_t sort_bytes = rk_sort_workspace_size(n, 8);
  void* sort_ws = ar.take<char>(sort_bytes);
  if (!keys || !hw_ok || !sort_ws) return RK_ERROR_WORKSPACE;
  const uint4* f = reinterpret_cast<const uint4*>(faces);
  const float4* v = reinterpret_cast<const float4*>(vertices);
  uint32_t* order = bvh->indices;
  RkSortPlan<uint64_t> plan;
  rk_status s = rk_sort_plan<uint64_t>(n, key_bits_for(mesh_count), true, keys, order, sort_ws, sort_bytes, plan);
  if (s != RK_SUCCESS) return s;
  if ((s = rk_fill_u32(stream, info, RK_INFO_WORDS, 0u)) != RK_SUCCESS) return s;
  hipLaunchKernelGGL(k_batch_prep, dim3(blocks_for(n, 256)), dim3(256), 0, st, meshes, mesh_count, f, v, n, hitboxes,
                     plan.src, plan.vsrc);
  RK_CHECK_LAUNCH();
  s = rk_sort_run<uint64_t>(st, plan, false, info + RK_INFO_FLAGS);
  if (s != RK_SUCCESS) return s;
  return launch_hierarchy<uint64_t, true>(st, keys, order, f, v, n, config->leaf_max, hw,
                                          static_cast<FNode*>(bvh->nodes), static_cast<float4*>(bvh->tris), meshes);
}

extern "C" size_t rk_batch_trace_workspace_size(uint32_t mesh_count, uint32_t ray_count) {
  (void)mesh_count;
  const size_t n = ray_count ? ray_count : 1;
  // the flags word, the queue counters, then (ray_order 1) the ray keys, the ray
  // order and the sort's own space
  return rk_align_up(4) + rk_align_up(kQueues * kQueueStride * 4) + rk_align_up(n * 8) + rk_align_up(n * 4) +
         rk_sort_workspace_size((uint32_t)n, 8) + 1024;
}

template <int kWG, int kStackN, int kDM>
static void launch_batch_trace(hipStream_t st, uint32_t mode, uint32_t grid_persistent, const rk_batch_mesh* meshes,
                               uint32_t mesh_count, const FNode* nodes, const float4* tris, uint32_t n_tris,
                               const float4* o, const float4* d, uint32_t n_rays, uint32_t* fid, float2* uv,
                               float* dep, float eps, uint32_t* queues, const uint32_t* order) {
  if (mode == 0)
    hipLaunchKernelGGL((k_batch_trace_grid<kWG, kStackN, kDM>), dim3(blocks_for(n_rays, kWG)), dim3(kWG), 0, st, meshes,
                       mesh_count, nodes, tris, n_tris, o, d, n_rays, fid, uv, dep, eps, order);
  else
    hipLaunchKernelGGL((k_batch_trace_queue<kWG, kStackN, kDM>), dim3(grid_persistent), dim3(kWG), 0, st, meshes,
                       mesh_count, nodes, tris, n_tris, o, d, n_rays, fid, uv, dep, eps, queues, order);
}

static inline float batch_eps_of(const rk_trace_options* o) {
  return o ? o->det_epsilon : RK_DET_EPSILON_REFERENCE;
}

extern "C" rk_status rk_batch_trace(rk_stream stream, const rk_batch_mesh* meshes, uint32_t mesh_count,
                                    const rk_fast_bvh* bvh, const rk_float4* origins, const rk_float4* directions,
                                    uint32_t ray_count, uint32_t* faces_id, rk_float2* coords, float* depths,
                                    const rk_trace_options* options, const rk_batch_config* config, void* ws,
                                    size_t ws_bytes) {
  if (!meshes || mesh_count == 0 || mesh_count > RK_BATCH_MAX_MESHES || !bvh || !bvh->nodes || !bvh->tris ||
      bvh->face_count == 0 || !config_ok(config))
    return RK_ERROR_INVALID_VALUE;
  if (ray_count == 0) return RK_SUCCESS;
  if (!origins || !directions || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  RkArena ar(ws, ws_bytes);
  uint32_t* flags = ar.take<uint32_t>(1);  // word 0 of ws: RK_FLAG_* bits of this call
  uint32_t* queues = ar.take<uint32_t>(kQueues * kQueueStride);
  if (!flags || !queues) return RK_ERROR_WORKSPACE;
  {
    rk_status s = rk_fill_u32(stream, flags, 1, 0u);
    if (s != RK_SUCCESS) return s;
  }
  uint32_t grid_persistent = 0;
  if (config->trace_mode == 1) {
    rk_status s = rk_fill_u32(stream, queues, kQueues * kQueueStride, 0u);
    if (s != RK_SUCCESS) return s;
    int dev = 0, cus = 0;
    RK_HIP(hipGetDevice(&dev));
    RK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // As many waves as are resident at once (20 per CU; the 1024-mesh batch takes 3.99
    // ms, with 16 per CU 4.12, 32 3.99), no more than there are tiles (100 meshes of at
    // most 4096 rays: without this limit 0.06 ms more), in a multiple of the eight XCDs.
    const uint32_t waves = std::min((uint32_t)cus * 20u, blocks_for(ray_count, 64));
    grid_persistent = blocks_for(waves, config->trace_wg / 64);
    grid_persistent = (grid_persistent + kQueues - 1) / kQueues * kQueues;
  }
  const FNode* nodes = static_cast<const FNode*>(bvh->nodes);
  const float4* tris = static_cast<const float4*>(bvh->tris);
  const float4* o = reinterpret_cast<const float4*>(origins);
  const float4* d = reinterpret_cast<const float4*>(directions);
  float2* uv = reinterpret_cast<float2*>(coords);
  const float eps = batch_eps_of(options);
  const uint32_t nt = bvh->face_count, mode = config->trace_mode;
  uint32_t* order = nullptr;
  if (config->ray_order == 1) {
    uint64_t* keys = ar.take<uint64_t>(ray_count);
    order = ar.take<uint32_t>(ray_count);
    const size_t sort_bytes = rk_sort_workspace_size(ray_count, 8);
    void* sort_ws = ar.take<char>(sort_bytes);
    if (!keys || !order || !sort_ws) return RK_ERROR_WORKSPACE;
    RkSortPlan<uint64_t> plan;
    rk_status s = rk_sort_plan<uint64_t>(ray_count, key_bits_for(mesh_count), true, keys, order, sort_ws, sort_bytes,
                                         plan);
    if (s != RK_SUCCESS) return s;
    hipLaunchKernelGGL(k_batch_ray_keys, dim3(blocks_for(ray_count, 256)), dim3(256), 0, st, meshes, mesh_count,
                       nodes, o, ray_count, plan.src, plan.vsrc);
    RK_CHECK_LAUNCH();
    s = rk_sort_run<uint64_t>(st, plan, false, flags);
    if (s != RK_SUCCESS) return s;
  }
#define RK_BATCH_TRACE(WG, SD, DM)                                                                                 \
  launch_batch_trace<WG, SD, DM>(st, mode, grid_persistent, meshes, mesh_count, nodes, tris, nt, o, d, ray_count,  \
                                 faces_id, uv, depths, eps, queues, order)
#define RK_BATCH_TRACE_DM(WG, SD)                        \
  do {                                                   \
    if (dm32) RK_BATCH_TRACE(WG, SD, 32);                \
    else RK_BATCH_TRACE(WG, SD, kTraceDonateMin);        \
  } while (0)
  const bool deep = config->stack_depth == 96, dm32 = config->donate_min == 32;
  switch (config->trace_wg) {
    case 64: if (deep) RK_BATCH_TRACE_DM(64, 96); else RK_BATCH_TRACE_DM(64, 64); break;
    case 128: if (deep) RK_BATCH_TRACE_DM(128, 96); else RK_BATCH_TRACE_DM(128, 64); break;
    default: if (deep) RK_BATCH_TRACE_DM(256, 96); else RK_BATCH_TRACE_DM(256, 64); break;
  }
#undef RK_BATCH_TRACE_DM
#undef RK_BATCH_TRACE
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

static inline float det_eps_of(const rk_trace_options* o) {
  return o ? o->det_epsilon : RK_DET_EPSILON_REFERENCE;
}
static inline uint32_t trace_flags_of(const rk_trace_options* o) { return o ? (o->flags & RK_TRACE_RESET_DEPTH) : 0u; }


extern "C" rk_status rk_fast_trace_counted(rk_stream stream, const rk_fast_bvh* bvh, const rk_float4* origins,
                                           const rk_float4* directions, uint32_t n_rays, uint32_t* faces_id,
                                           rk_float2* coords, float* depths, const rk_trace_options* options,
                                           uint64_t* counters) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0 || !counters) return RK_ERROR_INVALID_VALUE;
  if (n_rays == 0) return RK_SUCCESS;
  if (!origins || !directions || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL((k_fast_trace_v<true, kTraceWG, kSpreadRun, kLdsStack, false, 0, kTraceDonateMin>), dim3(blocks_for(n_rays, kTraceWG)), dim3(kTraceWG), 0, rk_hip_stream(stream),
                     static_cast<const FNode*>(bvh->nodes), static_cast<const float4*>(bvh->tris), bvh->face_count,
                     reinterpret_cast<const float4*>(origins), reinterpret_cast<const float4*>(directions), n_rays,
                     faces_id, reinterpret_cast<float2*>(coords), depths, det_eps_of(options),
                     reinterpret_cast<unsigned long long*>(counters), (const uint32_t*)nullptr, trace_flags_of(options));
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

// ---- camera frames, deformation, frame checksums --------------------------------

namespace {

// Bands of the camera kernel: 8 bands of 8-pixel runs measured best on the
// 1920x1080 heightfield frame (with help at one idle lane 0.173 ms; 16 bands of
// 4-pixel runs 0.195, 4 bands 0.176; with the default's 16 idle lanes 0.163).
#ifndef RK_CAM_BANDS
#define RK_CAM_BANDS 8
#endif
constexpr int kCamBands = RK_CAM_BANDS, kCamRun = 64 / RK_CAM_BANDS;
static_assert(kCamBands >= 1 && 64 % kCamBands == 0, "runs tile a wave");

__device__ __forceinline__ uint64_t mix64(uint64_t z) {  // SplitMix64 finaliser
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ float u01_of(uint64_t h) { return (float)(h >> 40) * (1.0f / 16777216.0f); }

// v = base + amplitude * sin(omega * time + phase_v) * axis_v; phase and axis
// hashed from the vertex index (axis uniform on the sphere, or +z).
__global__ __launch_bounds__(256) void k_deform(const float4* __restrict__ base, float4* __restrict__ out,
                                                uint32_t count, float amplitude, float omega, float time,
                                                uint64_t seed, int along_z) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const uint64_t h0 = mix64(seed ^ (0x9E3779B97F4A7C15ull * ((uint64_t)i + 1)));
  const uint64_t h1 = mix64(h0 + 0x632BE59BD9B4E019ull), h2 = mix64(h1 + 0x632BE59BD9B4E019ull);
  const float phase = 6.2831853f * u01_of(h0);
  float ax = 0.0f, ay = 0.0f, az = 1.0f;
  if (!along_z) {
    const float z = 2.0f * u01_of(h1) - 1.0f, phi = 6.2831853f * u01_of(h2);
    const float r = sqrtf(fmaxf(0.0f, 1.0f - z * z));
    ax = r * cosf(phi);
    ay = r * sinf(phi);
    az = z;
  }
  const float s = amplitude * sinf(omega * time + phase);
  const float4 b = base[i];
  out[i] = make_float4(b.x + s * ax, b.y + s * ay, b.z + s * az, b.w);
}

__device__ __forceinline__ uint64_t shfl_down64(uint64_t v, int d) {
  uint32_t lo = __shfl_down((uint32_t)v, d, 64), hi = __shfl_down((uint32_t)(v >> 32), d, 64);
  return ((uint64_t)hi << 32) | lo;
}

// Order-independent frame checksum: the wrapping sum over rays of a hash of
// (ray, original face id, depth, u, v bits), and the hit count. Original ids
// make it independent of the tree the frame was traced with. A fixed grid of
// at most kSumBlocks workgroups walks the frame, reduces in registers, waves
// and LDS, and adds once per workgroup: same-address atomics from every wave
// would serialise across XCDs.
constexpr uint32_t kSumBlocks = 256;
static_assert(kSumBlocks <= 256, "k_checksum_to_host's last workgroup reads one share per thread");

// One ray's term of the frame checksum.
__device__ __forceinline__ uint64_t ray_hash(uint32_t i, uint32_t orig, float depth, float2 c) {
  return mix64(((uint64_t)i << 32 | orig) ^ mix64(((uint64_t)__float_as_uint(depth) << 32) ^
                                                  ((uint64_t)__float_as_uint(c.x) * 0x100000001B3ull) ^
                                                  __float_as_uint(c.y)));
}

// Wave and workgroup sums of (h, n), valid in thread 0 of the workgroup.
__device__ __forceinline__ void block_sum2(uint64_t& h, uint64_t& n) {
  __shared__ uint64_t s_h[4], s_n[4];
  for (int d = 32; d >= 1; d >>= 1) {  // lane 0 ends with the wave's sums
    h += shfl_down64(h, d);
    n += shfl_down64(n, d);
  }
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { s_h[w] = h; s_n[w] = n; }
  __syncthreads();
  h = s_h[0] + s_h[1] + s_h[2] + s_h[3];
  n = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

// This workgroup's share of the frame checksum: (hash sum, hits), valid in thread 0.
__device__ __forceinline__ void block_checksum(const uint32_t* __restrict__ faces_id,
                                               const float2* __restrict__ coords, const float* __restrict__ depths,
                                               uint32_t count, const uint32_t* __restrict__ indices,
                                               uint32_t n_faces, uint64_t& bh, uint64_t& bn) {
  uint64_t h = 0, hit = 0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
    const uint32_t f = faces_id[i];
    const bool is_hit = f != 0xFFFFFFFFu && f < n_faces;
    h += ray_hash(i, is_hit ? (indices ? indices[f] : f) : 0xFFFFFFFFu, depths[i], coords[i]);
    hit += is_hit ? 1 : 0;
  }
  block_sum2(h, hit);
  bh = h;
  bn = hit;
}

__global__ __launch_bounds__(256) void k_checksum(const uint32_t* __restrict__ faces_id,
                                                  const float2* __restrict__ coords,
                                                  const float* __restrict__ depths, uint32_t count,
                                                  const uint32_t* __restrict__ indices, uint32_t n_faces,
                                                  unsigned long long* __restrict__ out) {
  uint64_t bh, bn;
  block_checksum(faces_id, coords, depths, count, indices, n_faces, bh, bn);
  if (threadIdx.x == 0) {
    atomicAdd(out, (unsigned long long)bh);
    atomicAdd(out + 1, (unsigned long long)bn);
  }
}

// The end of a one-launch checksum, called by every thread of every
// workgroup with the workgroup's share in thread 0 (bh, bn): each workgroup
// stores its share in partials (2 words each), and the last one to count
// itself in adds the shares, writes the total to out[0..1] (host memory
// mapped for the device), sets the counter back to zero for the next launch,
// and then writes done_value to out[2]: the host sees the frame finished
// without a runtime query.
// out[0] = hash sum, out[1] = hits; with build_flags, out[3] = *build_flags;
// out[2] = done_value last.
__device__ __forceinline__ void finish_checksum(uint64_t bh, uint64_t bn, uint64_t* __restrict__ partials,
                                                uint32_t* __restrict__ counter, uint64_t* out, uint64_t done_value,
                                                const uint32_t* build_flags = nullptr) {
  __shared__ uint32_t s_last;
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = bh;
    partials[2 * blockIdx.x + 1] = bn;
    __threadfence();
    s_last = atomicAdd(counter, 1u) == gridDim.x - 1 ? 1u : 0u;
  }
  __syncthreads();
  if (!s_last) return;  // workgroup-uniform
  __threadfence();
  uint64_t h = 0, n = 0;
  for (uint32_t b = threadIdx.x; b < gridDim.x; b += blockDim.x) {
    h += __hip_atomic_load(partials + 2 * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    n += __hip_atomic_load(partials + 2 * b + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  for (int d = 32; d >= 1; d >>= 1) {
    h += shfl_down64(h, d);
    n += shfl_down64(n, d);
  }
  __shared__ uint64_t s_h[4], s_n[4];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { s_h[w] = h; s_n[w] = n; }
  __syncthreads();
  if (threadIdx.x == 0) {
    out[0] = s_h[0] + s_h[1] + s_h[2] + s_h[3];
    out[1] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
    if (build_flags) out[3] = __hip_atomic_load(build_flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *counter = 0u;
    __threadfence_system();  // the total lands before the done word
    __hip_atomic_store(out + 2, done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// The checksum of a frame in memory in one launch (finish_checksum).
__global__ __launch_bounds__(256) void k_checksum_to_host(const uint32_t* __restrict__ faces_id,
                                                          const float2* __restrict__ coords,
                                                          const float* __restrict__ depths, uint32_t count,
                                                          const uint32_t* __restrict__ indices, uint32_t n_faces,
                                                          uint64_t* __restrict__ partials,
                                                          uint32_t* __restrict__ counter, uint64_t* out,
                                                          uint64_t done_value, const uint32_t* build_flags) {
  uint64_t bh, bn;
  block_checksum(faces_id, coords, depths, count, indices, n_faces, bh, bn);
  finish_checksum(bh, bn, partials, counter, out, done_value, build_flags);
}

// Which pixel a camera-kernel lane traces. Wave g takes a row segment of
// 64 / kBands pixels in each of kBands horizontal bands of the image, at the
// same place in every band, for the reason given at spread_ray.
//
// With kXcd, workgroups are dealt to the eight XCDs round-robin (block b runs
// on XCD b mod 8), and XCD x takes the x-th of eight vertical strips of the
// image: its L2 then holds the nodes of one eighth of the view, where each L2
// would otherwise fetch the nodes of the whole view. The waves of a strip are
// taken row segment by row segment; the horizon, which crosses every strip,
// spreads over all eight. Blocks past a strip's waves have no pixels.
template <int kWG, int kBands, bool kXcd>
__device__ __forceinline__ bool camera_pixel(int width, int height, int& x, int& y) {
  constexpr int kRun = 64 / kBands;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int segs = (width + kRun - 1) / kRun, band_h = (height + kBands - 1) / kBands;
  int seg, row_in_band;
  if (kXcd) {
    const int sw = (segs + 7) / 8;  // segments per strip
    const int xcd = blockIdx.x & 7;
    const int w = (int)(blockIdx.x >> 3) * (kWG / 64) + wave;
    seg = xcd * sw + w % sw;
    row_in_band = seg < segs ? w / sw : band_h;  // the last strip can be narrower
  } else {
    const int g = (int)blockIdx.x * (kWG / 64) + wave;
    seg = g % segs;
    row_in_band = g / segs;
  }
  x = seg * kRun + lane % kRun;
  y = (lane / kRun) * band_h + row_in_band;
  return row_in_band < band_h && x < width && y < height;
}

// Primary ray of pixel (x, y) generated in the trace kernel itself (the
// reference's CUDA_calcPrimaryRays.cu:43-55 formula: origin, and direction
// (dir - x * step_x) - y * step_y), so a frame reads no ray arrays. Every pixel is written:
// a miss gives face ~0, coords (0, 0), depth FLT_MAX.
template <int kWG, int kBands, bool kXcd, bool kOldest = false, int kLeafBatch = 0, int kDonateMin = 1>
__global__ __launch_bounds__(kWG) void k_fast_trace_camera_v(const FNode* __restrict__ nodes,
                                                             const float4* __restrict__ tris, uint32_t n_tris,
                                                             float4 ro, float4 rd, float4 rx, float4 ry, int width,
                                                             int height, uint32_t* __restrict__ faces_id,
                                                             float2* __restrict__ coords, float* __restrict__ depths,
                                                             float eps) {
  int x, y;
  const bool has_ray = camera_pixel<kWG, kBands, kXcd>(width, height, x, y);
  const float4 d = rk::sub4(rk::sub4(rd, rk::muls4(rx, (float)x)), rk::muls4(ry, (float)y));
  uint32_t nb = 0, nt = 0;
  __shared__ uint2 s_stack[kLdsStack * kWG];
  __shared__ uint32_t s_xchg[kWG / 64][kXchgWords];
  const RayHit h = trace_ray_shared<false, kStack, kLdsStack, kWG, kOldest, kLeafBatch, kDonateMin>(
      nodes, tris, n_tris, 0u, has_ray, ro, d,
                                                                            RK_HUGE, eps, nb, nt, s_stack,
                                                                            s_xchg[threadIdx.x >> 6]);
  if (!has_ray) return;
  const size_t p = (size_t)y * (size_t)width + (size_t)x;
  const bool hit = h.pos != 0xFFFFFFFFu;
  faces_id[p] = h.pos;
  coords[p] = hit ? make_float2(h.u, h.v) : make_float2(0.0f, 0.0f);
  depths[p] = hit ? h.t : RK_HUGE;
}

// The sample-02 frame in one launch: each pixel's primary ray, its closest hit
// (as k_fast_trace_camera_v), the hit face's normal at (u, v) (as
// rk_interpolate_data) and the pixel (as rk_shade), with the same arithmetic in
// the same order as those three kernels, so the pixels are bit-identical to
// theirs. faces: the mesh's faces in the tree's leaf order (faces[position]),
// as the reference's builds leave them. faces_id, coords and depths, when not
// NULL, receive what k_fast_trace_camera_v writes.
template <int kWG, int kBands, int kDM>
__global__ __launch_bounds__(kWG) void k_fast_render_camera(
    const FNode* __restrict__ nodes, const float4* __restrict__ tris, uint32_t n_tris, float4 ro, float4 rd,
    float4 rx, float4 ry, int width, int height, const uint4* __restrict__ faces, const float4* __restrict__ verts,
    const float4* __restrict__ norms, float4 back, float4 cam, uint32_t* __restrict__ pixels, int pitch,
    uint32_t* __restrict__ faces_id, float2* __restrict__ coords, float* __restrict__ depths, float eps) {
  int x, y;
  const bool has_ray = camera_pixel<kWG, kBands, false>(width, height, x, y);
  const float4 d = rk::sub4(rk::sub4(rd, rk::muls4(rx, (float)x)), rk::muls4(ry, (float)y));
  uint32_t nb = 0, nt = 0;
  __shared__ uint2 s_stack[kLdsStack * kWG];
  __shared__ uint32_t s_xchg[kWG / 64][kXchgWords];
  const RayHit h = trace_ray_shared<false, kStack, kLdsStack, kWG, false, 0, kDM>(
      nodes, tris, n_tris, 0u, has_ray, ro, d, RK_HUGE, eps, nb, nt, s_stack, s_xchg[threadIdx.x >> 6]);
  if (!has_ray) return;
  const bool hit = h.pos != 0xFFFFFFFFu;  // then t < FLT_MAX: the shader's depth test
  if (faces_id) {
    const size_t p = (size_t)y * (size_t)width + (size_t)x;
    faces_id[p] = h.pos;
    coords[p] = hit ? make_float2(h.u, h.v) : make_float2(0.0f, 0.0f);
    depths[p] = hit ? h.t : RK_HUGE;
  }
  pixels[(size_t)y * (size_t)pitch + (size_t)x] =
      hit ? rk::shade_hit(cam, rk::face_normal_at(faces[h.pos], h.u, h.v, verts, norms)) : rk::make_pixel(back);
}

// Workgroups of a camera-kernel variant for a width x height frame.
uint32_t camera_blocks(int width, int height, int wg, int bands, bool xcd) {
  const int run = 64 / bands;
  const uint64_t segs = (uint64_t)((width + run - 1) / run), band_h = (uint64_t)((height + bands - 1) / bands);
  const uint64_t wpb = (uint64_t)(wg / 64);
  if (xcd) {
    const uint64_t sw = (segs + 7) / 8;
    return (uint32_t)(8 * ((sw * band_h + wpb - 1) / wpb));
  }
  return (uint32_t)((segs * band_h + wpb - 1) / wpb);
}

}  // namespace

// ---- traversal variants and the autotuner ------------------------------------------
namespace {

typedef void (*TraceKernel)(const FNode*, const float4*, uint32_t, const float4*, const float4*, uint32_t, uint32_t*,
                            float2*, float*, float, unsigned long long*, const uint32_t*, uint32_t);
typedef void (*CameraKernel)(const FNode*, const float4*, uint32_t, float4, float4, float4, float4, int, int,
                             uint32_t*, float2*, float*, float);
struct TraceVariant {
  uint32_t wg, run, lds, oldest, leaf_batch, donate_min, bound_every;
  TraceKernel kernel;
};
struct CameraVariant {
  uint32_t wg, bands, xcd, oldest, leaf_batch, donate_min;
  CameraKernel kernel;
};

// rk_trace_options.config k selects entry k - 1 (0: the first, or one that is not listed
// by the sizes, in rk_fast_trace and rk_fast_trace_sorted). All fetch together; for rays
// that share no nodes those that postpone leaves come out best (2M on 300,000 faces 1.90 ms).
#define RK_TRACE_VARIANT(wg, run, lds, old, lb, dm) \
  {wg, run, lds, old, lb, dm, 1, k_fast_trace_v<false, wg, run, lds, old != 0, lb, dm>}
#define RK_TRACE_VARIANT_B(dm, be) {64, 8, 8, 0, 0, dm, be, k_fast_trace_v<false, 64, 8, 8, false, 0, dm, be>}

const TraceVariant kTraceVariants[] = {
    RK_TRACE_VARIANT(kTraceWG, kSpreadRun, kLdsStack, 0, 0, kTraceDonateMin),
    RK_TRACE_VARIANT(64, 4, 8, 0, 0, 1),   RK_TRACE_VARIANT(64, 16, 8, 0, 0, 1), RK_TRACE_VARIANT(64, 0, 8, 0, 0, 1),
    RK_TRACE_VARIANT(64, 8, 4, 0, 0, 1),   RK_TRACE_VARIANT(64, 8, 12, 0, 0, 1), RK_TRACE_VARIANT(128, 8, 8, 0, 0, 1),
    RK_TRACE_VARIANT(128, 16, 8, 0, 0, 1), RK_TRACE_VARIANT(256, 8, 8, 0, 0, 1), RK_TRACE_VARIANT(64, 8, 8, 1, 0, 1),
    RK_TRACE_VARIANT(64, 4, 8, 1, 0, 1),   RK_TRACE_VARIANT(64, 0, 8, 1, 0, 1),  RK_TRACE_VARIANT(128, 8, 8, 1, 0, 1),
    RK_TRACE_VARIANT(64, 8, 8, 0, 8, 1),   RK_TRACE_VARIANT(64, 8, 8, 0, 16, 1), RK_TRACE_VARIANT(64, 8, 8, 0, 32, 1),
    RK_TRACE_VARIANT(64, 8, 8, 0, 0, 8),   RK_TRACE_VARIANT(64, 8, 8, 0, 0, 1),  RK_TRACE_VARIANT(64, 8, 8, 0, 16, 8),
    RK_TRACE_VARIANT(64, 8, 8, 0, 16, 16), RK_TRACE_VARIANT(64, 8, 8, 0, 32, 16), RK_TRACE_VARIANT(64, 8, 8, 0, 0, 32),
    RK_TRACE_VARIANT(64, 8, 8, 1, 0, 16),
    RK_TRACE_VARIANT_B(16, 2),             RK_TRACE_VARIANT_B(16, 4),            RK_TRACE_VARIANT_B(32, 2),
    RK_TRACE_VARIANT_B(32, 4),
};
#undef RK_TRACE_VARIANT
#undef RK_TRACE_VARIANT_B
#define RK_CAMERA_VARIANT(wg, bands, xcd, old, lb, dm) \
  {wg, bands, xcd, old, lb, dm, k_fast_trace_camera_v<wg, bands, xcd != 0, old != 0, lb, dm>}
const CameraVariant kCameraVariants[] = {
    RK_CAMERA_VARIANT(kTraceWG, kCamBands, 0, 0, 0, kTraceDonateMin),
    RK_CAMERA_VARIANT(64, 8, 1, 0, 0, 1),   RK_CAMERA_VARIANT(64, 4, 0, 0, 0, 1),   RK_CAMERA_VARIANT(64, 4, 1, 0, 0, 1),
    RK_CAMERA_VARIANT(64, 16, 0, 0, 0, 1),  RK_CAMERA_VARIANT(64, 16, 1, 0, 0, 1),  RK_CAMERA_VARIANT(128, 8, 0, 0, 0, 1),
    RK_CAMERA_VARIANT(128, 8, 1, 0, 0, 1),  RK_CAMERA_VARIANT(128, 16, 0, 0, 0, 1), RK_CAMERA_VARIANT(128, 16, 1, 0, 0, 1),
    RK_CAMERA_VARIANT(64, 8, 0, 1, 0, 1),   RK_CAMERA_VARIANT(64, 4, 0, 1, 0, 1),   RK_CAMERA_VARIANT(128, 8, 0, 1, 0, 1),
    RK_CAMERA_VARIANT(64, 8, 1, 1, 0, 1),   RK_CAMERA_VARIANT(64, 8, 0, 0, 16, 1),  RK_CAMERA_VARIANT(64, 8, 0, 0, 32, 1),
    RK_CAMERA_VARIANT(64, 8, 0, 0, 16, 16), RK_CAMERA_VARIANT(64, 8, 0, 0, 0, 1),   RK_CAMERA_VARIANT(64, 8, 0, 0, 0, 32),
    RK_CAMERA_VARIANT(128, 8, 0, 1, 0, 16),
};
#undef RK_CAMERA_VARIANT
constexpr uint32_t kNumTraceVariants = sizeof(kTraceVariants) / sizeof(kTraceVariants[0]);
constexpr uint32_t kNumCameraVariants = sizeof(kCameraVariants) / sizeof(kCameraVariants[0]);

const TraceVariant* trace_variant(uint32_t config) {
  return config == 0 ? &kTraceVariants[0] : (config <= kNumTraceVariants ? &kTraceVariants[config - 1] : nullptr);
}
const CameraVariant* camera_variant(uint32_t config) {
  return config == 0 ? &kCameraVariants[0] : (config <= kNumCameraVariants ? &kCameraVariants[config - 1] : nullptr);
}

rk_status launch_trace_variant(hipStream_t st, const TraceVariant& tv, const rk_fast_bvh* bvh,
                               const rk_float4* origins, const rk_float4* directions, uint32_t n_rays,
                               uint32_t* faces_id, rk_float2* coords, float* depths, float eps, uint32_t flags) {
  hipLaunchKernelGGL(tv.kernel, dim3(blocks_for(n_rays, tv.wg)), dim3(tv.wg), 0, st,
                     static_cast<const FNode*>(bvh->nodes), static_cast<const float4*>(bvh->tris), bvh->face_count,
                     reinterpret_cast<const float4*>(origins), reinterpret_cast<const float4*>(directions), n_rays,
                     faces_id, reinterpret_cast<float2*>(coords), depths, eps, (unsigned long long*)nullptr,
                     (const uint32_t*)nullptr, flags);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

void describe_trace(uint32_t config, rk_trace_tuning* out) {
  const TraceVariant& v = *trace_variant(config);
  *out = rk_trace_tuning{};
  out->config = config;
  out->workgroup = v.wg;
  out->ray_run = v.run;
  out->lds_stack = v.lds;
  out->steal_oldest = v.oldest;
  out->leaf_batch = v.leaf_batch;
  out->donate_min = v.donate_min;
  out->bound_every = v.bound_every;
}
void describe_camera(uint32_t config, rk_trace_tuning* out) {
  const CameraVariant& v = *camera_variant(config);
  *out = rk_trace_tuning{};
  out->config = config;
  out->workgroup = v.wg;
  out->ray_run = 64 / v.bands;
  out->bands = v.bands;
  out->lds_stack = kLdsStack;
  out->xcd_strips = v.xcd;
  out->steal_oldest = v.oldest;
  out->leaf_batch = v.leaf_batch;
  out->donate_min = v.donate_min;
  out->bound_every = 1;
}

// Times fn() reps times after one untimed call, each call preceded by
// prep() outside the timed region; returns the mean in ms.
template <typename Prep, typename Fn>
rk_status time_calls(hipStream_t st, hipEvent_t e0, hipEvent_t e1, int reps, Prep prep, Fn fn, float* ms) {
  float total = 0.0f;
  for (int r = 0; r <= reps; ++r) {
    rk_status s = prep();
    if (s != RK_SUCCESS) return s;
    RK_HIP(hipEventRecord(e0, st));
    s = fn();
    if (s != RK_SUCCESS) return s;
    RK_HIP(hipEventRecord(e1, st));
    RK_HIP(hipEventSynchronize(e1));
    float t = 0.0f;
    RK_HIP(hipEventElapsedTime(&t, e0, e1));
    if (r > 0) total += t;
  }
  *ms = total / (float)reps;
  return RK_SUCCESS;
}

struct EventPair {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  ~EventPair() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
  }
};

}  // namespace

extern "C" rk_status rk_fast_trace_variant(uint32_t config, int camera, rk_trace_tuning* out) {
  if (!out) return RK_ERROR_INVALID_VALUE;
  if (camera ? !camera_variant(config) : !trace_variant(config)) return RK_ERROR_INVALID_VALUE;
  if (camera)
    describe_camera(config, out);
  else
    describe_trace(config, out);
  return RK_SUCCESS;
}

extern "C" size_t rk_fast_autotune_workspace_size(uint32_t n_rays) {
  return rk_align_up((size_t)(n_rays ? n_rays : 1) * 4) + 256;
}

extern "C" rk_status rk_fast_autotune(rk_stream stream, const rk_fast_bvh* bvh, const rk_float4* origins,
                                      const rk_float4* directions, uint32_t n_rays, uint32_t* faces_id,
                                      rk_float2* coords, float* depths, const rk_trace_options* options, int reps,
                                      void* ws, size_t ws_bytes, rk_trace_tuning* best) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0 || !best) return RK_ERROR_INVALID_VALUE;
  if (n_rays == 0 || !origins || !directions || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  if (reps < 1 || reps > 100) return RK_ERROR_INVALID_VALUE;
  if (!ws || ws_bytes < rk_fast_autotune_workspace_size(n_rays)) return RK_ERROR_WORKSPACE;
  hipStream_t st = rk_hip_stream(stream);
  const float eps = det_eps_of(options);
  float* tmax = static_cast<float*>(ws);
  RK_HIP(hipMemcpyAsync(tmax, depths, 4ull * n_rays, hipMemcpyDeviceToDevice, st));
  EventPair ev;
  RK_HIP(hipEventCreate(&ev.e0));
  RK_HIP(hipEventCreate(&ev.e1));
  // with RK_TRACE_RESET_DEPTH the calls do not read depths: nothing to restore
  const bool reset = (trace_flags_of(options) & RK_TRACE_RESET_DEPTH) != 0u;
  auto restore = [&]() -> rk_status {
    if (!reset) RK_HIP(hipMemcpyAsync(depths, tmax, 4ull * n_rays, hipMemcpyDeviceToDevice, st));
    return RK_SUCCESS;
  };
  uint32_t best_cfg = 0;
  float best_ms = 0.0f;
  for (uint32_t k = 0; k < kNumTraceVariants; ++k) {
    float ms = 0.0f;
    const TraceVariant& tv = kTraceVariants[k];
    rk_status s = time_calls(st, ev.e0, ev.e1, reps, restore, [&]() {
      return launch_trace_variant(st, tv, bvh, origins, directions, n_rays, faces_id, coords, depths, eps,
                                  trace_flags_of(options));
    }, &ms);
    if (s != RK_SUCCESS) return s;
    if (k == 0 || ms < best_ms) {
      best_ms = ms;
      best_cfg = k + 1;
    }
  }
  // leave the caller's frame traced by the chosen variant
  rk_status s = restore();
  if (s != RK_SUCCESS) return s;
  s = launch_trace_variant(st, *trace_variant(best_cfg), bvh, origins, directions, n_rays, faces_id, coords, depths,
                           eps, trace_flags_of(options));
  if (s != RK_SUCCESS) return s;
  describe_trace(best_cfg, best);
  best->ms = best_ms;
  return RK_SUCCESS;
}

extern "C" rk_status rk_fast_autotune_camera(rk_stream stream, const rk_fast_bvh* bvh, const rk_camera_rays* camera,
                                             int width, int height, uint32_t* faces_id, rk_float2* coords,
                                             float* depths, const rk_trace_options* options, int reps,
                                             rk_trace_tuning* best) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0 || !camera || !best) return RK_ERROR_INVALID_VALUE;
  if (width <= 0 || height <= 0 || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  if ((uint64_t)width * (uint64_t)height > 0xFFFFFFFFull) return RK_ERROR_UNSUPPORTED;
  if (reps < 1 || reps > 100) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  EventPair ev;
  RK_HIP(hipEventCreate(&ev.e0));
  RK_HIP(hipEventCreate(&ev.e1));
  rk_trace_options opt = options ? *options : rk_trace_options{RK_DET_EPSILON_REFERENCE, 0u, 0u, 0u};
  uint32_t best_cfg = 0;
  float best_ms = 0.0f;
  for (uint32_t k = 0; k < kNumCameraVariants; ++k) {
    float ms = 0.0f;
    opt.config = k + 1;
    rk_status s = time_calls(st, ev.e0, ev.e1, reps, []() { return (rk_status)RK_SUCCESS; }, [&]() {
      return rk_fast_trace_camera(stream, bvh, camera, width, height, faces_id, coords, depths, &opt);
    }, &ms);
    if (s != RK_SUCCESS) return s;
    if (k == 0 || ms < best_ms) {
      best_ms = ms;
      best_cfg = k + 1;
    }
  }
  opt.config = best_cfg;
  rk_status s = rk_fast_trace_camera(stream, bvh, camera, width, height, faces_id, coords, depths, &opt);
  if (s != RK_SUCCESS) return s;
  describe_camera(best_cfg, best);
  best->ms = best_ms;
  return RK_SUCCESS;
}

extern "C" rk_status rk_fast_trace(rk_stream stream, const rk_fast_bvh* bvh, const rk_float4* origins,
                                   const rk_float4* directions, uint32_t n_rays, uint32_t* faces_id, rk_float2* coords,
                                   float* depths, const rk_trace_options* options) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0) return RK_ERROR_INVALID_VALUE;
  if (n_rays == 0) return RK_SUCCESS;
  if (!origins || !directions || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  const TraceVariant* tv = trace_variant(options ? options->config : 0u);
  if (!tv) return RK_ERROR_INVALID_VALUE;
  TraceVariant v = *tv;
  if ((!options || options->config == 0) && bvh->face_count >= kMemoryFaces)
    v.kernel = k_fast_trace_v<false, kTraceWG, kSpreadRun, kDeepestLdsStack, false, 0, 32>;
  return launch_trace_variant(rk_hip_stream(stream), v, bvh, origins, directions, n_rays, faces_id, coords, depths,
                              det_eps_of(options), trace_flags_of(options));
}

extern "C" rk_status rk_fast_trace_camera(rk_stream stream, const rk_fast_bvh* bvh, const rk_camera_rays* camera,
                                          int width, int height, uint32_t* faces_id, rk_float2* coords, float* depths,
                                          const rk_trace_options* options) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0 || !camera) return RK_ERROR_INVALID_VALUE;
  if (width <= 0 || height <= 0 || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  if ((uint64_t)width * (uint64_t)height > 0xFFFFFFFFull) return RK_ERROR_UNSUPPORTED;
  auto f4 = [](const rk_float4& v) { return make_float4(v.x, v.y, v.z, v.w); };
  const CameraVariant* cv = camera_variant(options ? options->config : 0u);
  if (!cv) return RK_ERROR_INVALID_VALUE;
  dim3 grid(camera_blocks(width, height, (int)cv->wg, (int)cv->bands, cv->xcd != 0));
  hipLaunchKernelGGL(cv->kernel, grid, dim3(cv->wg), 0, rk_hip_stream(stream), static_cast<const FNode*>(bvh->nodes),
                     static_cast<const float4*>(bvh->tris), bvh->face_count, f4(camera->origin),
                     f4(camera->direction), f4(camera->step_x), f4(camera->step_y), width, height, faces_id,
                     reinterpret_cast<float2*>(coords), depths, det_eps_of(options));
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" rk_status rk_fast_render_camera(rk_stream stream, const rk_fast_bvh* bvh, const rk_camera_rays* camera,
                                           int width, int height, const rk_uint4* faces, const rk_float4* vertices,
                                           const rk_float4* normals, rk_float4 back_color, rk_float4 cam_dir,
                                           uint32_t* pixels, int pitch, uint32_t* faces_id, rk_float2* coords,
                                           float* depths, const rk_trace_options* options) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0 || !camera || !faces || !vertices || !pixels)
    return RK_ERROR_INVALID_VALUE;
  if (width <= 0 || height <= 0 || pitch < width) return RK_ERROR_INVALID_VALUE;
  if ((faces_id || coords || depths) && !(faces_id && coords && depths)) return RK_ERROR_INVALID_VALUE;
  if ((uint64_t)width * (uint64_t)height > 0xFFFFFFFFull || (uint64_t)pitch * (uint64_t)height > 0xFFFFFFFFull)
    return RK_ERROR_UNSUPPORTED;
  auto f4 = [](const rk_float4& v) { return make_float4(v.x, v.y, v.z, v.w); };
  dim3 grid(camera_blocks(width, height, kTraceWG, kCamBands, false));
  hipLaunchKernelGGL((k_fast_render_camera<kTraceWG, kCamBands, kTraceDonateMin>), grid, dim3(kTraceWG), 0,
                     rk_hip_stream(stream), static_cast<const FNode*>(bvh->nodes),
                     static_cast<const float4*>(bvh->tris), bvh->face_count, f4(camera->origin),
                     f4(camera->direction), f4(camera->step_x), f4(camera->step_y), width, height,
                     reinterpret_cast<const uint4*>(faces), reinterpret_cast<const float4*>(vertices),
                     reinterpret_cast<const float4*>(normals), f4(back_color),
                     make_float4(cam_dir.x, cam_dir.y, cam_dir.z, 0.0f), pixels, pitch, faces_id,
                     reinterpret_cast<float2*>(coords), depths, det_eps_of(options));
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" rk_status rk_deform_vertices(rk_stream stream, const rk_float4* base, rk_float4* out, uint32_t count,
                                        float amplitude, float omega, float time, uint64_t seed, int along_z) {
  if (count == 0) return RK_SUCCESS;
  if (!base || !out) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL(k_deform, dim3(blocks_for(count, 256)), dim3(256), 0, rk_hip_stream(stream),
                     reinterpret_cast<const float4*>(base), reinterpret_cast<float4*>(out), count, amplitude, omega,
                     time, seed, along_z);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" rk_status rk_frame_checksum(rk_stream stream, const uint32_t* faces_id, const rk_float2* coords,
                                       const float* depths, uint32_t count, const uint32_t* indices,
                                       uint32_t face_count, uint64_t* out) {
  if (!out) return RK_ERROR_INVALID_VALUE;
  rk_status s = rk_fill_u32(stream, reinterpret_cast<uint32_t*>(out), 4, 0u);
  if (s != RK_SUCCESS || count == 0) return s;
  if (!faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL(k_checksum, dim3(std::min(blocks_for(count, 256), kSumBlocks)), dim3(256), 0,
                     rk_hip_stream(stream), faces_id,
                     reinterpret_cast<const float2*>(coords), depths, count, indices, face_count,
                     reinterpret_cast<unsigned long long*>(out));
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

// The frame checksum for the request loop: one launch, the total written to
// out_host[0..1], a device-writable mapping of pinned coherent host memory,
// then done_value to out_host[2]. partials holds 2 * kSumBlocks words and
// counter one word that is zero between launches (zero it once before the
// first).
rk_status rk_frame_checksum_to_host(hipStream_t st, const uint32_t* faces_id, const rk_float2* coords,
                                    const float* depths, uint32_t count, const uint32_t* indices,
                                    uint32_t face_count, uint64_t* partials, uint32_t* counter, uint64_t* out_host,
                                    uint64_t done_value, const uint32_t* build_flags) {
  if (!faces_id || !coords || !depths || !partials || !counter || !out_host) return RK_ERROR_INVALID_VALUE;
  hipLaunchKernelGGL(k_checksum_to_host, dim3(std::max(1u, std::min(blocks_for(count, 256), kSumBlocks))), dim3(256),
                     0, st, faces_id, reinterpret_cast<const float2*>(coords), depths, count, indices, face_count,
                     partials, counter, out_host, done_value, build_flags);
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" size_t rk_fast_trace_sorted_workspace_size(uint32_t n_rays) {
  const size_t n = n_rays ? n_rays : 1;
  return rk_align_up(n * 4) * 2 + rk_sort_workspace_size((uint32_t)n, 4) + 1024;
}

extern "C" rk_status rk_fast_trace_sorted(rk_stream stream, const rk_fast_bvh* bvh, const rk_float4* origins,
                                          const rk_float4* directions, uint32_t n_rays, uint32_t* faces_id,
                                          rk_float2* coords, float* depths, const rk_trace_options* options,
                                          void* ws, size_t ws_bytes) {
  if (!bvh || !bvh->nodes || !bvh->tris || bvh->face_count == 0) return RK_ERROR_INVALID_VALUE;
  if (n_rays == 0) return RK_SUCCESS;
  if (!origins || !directions || !faces_id || !coords || !depths) return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  RkArena ar(ws, ws_bytes);
  const size_t sort_bytes = rk_sort_workspace_size(n_rays, 4);
  void* sort_ws = ar.take<char>(sort_bytes);  // first: its word 0 is the sort's error word
  uint32_t* keys = ar.take<uint32_t>(n_rays);
  uint32_t* order = ar.take<uint32_t>(n_rays);
  if (!keys || !order || !sort_ws) return RK_ERROR_WORKSPACE;
  const FNode* nodes = static_cast<const FNode*>(bvh->nodes);
  const float4* o = reinterpret_cast<const float4*>(origins);
  const TraceVariant* tv = trace_variant(options ? options->config : 0u);
  if (!tv) return RK_ERROR_INVALID_VALUE;
  RkSortPlan<uint32_t> plan;
  rk_status s = rk_sort_plan<uint32_t>(n_rays, 30, true, keys, order, sort_ws, sort_bytes, plan);
  if (s != RK_SUCCESS) return s;
  hipLaunchKernelGGL(k_ray_keys, dim3(blocks_for(n_rays, 256)), dim3(256), 0, st, nodes, o, n_rays, plan.src,
                     plan.vsrc);
  RK_CHECK_LAUNCH();
  s = rk_sort_run<uint32_t>(st, plan, false, nullptr);
  if (s != RK_SUCCESS) return s;
  // the variant's workgroup, stack and exchange settings; the order replaces its ray runs
  const bool by_rule = !options || options->config == 0;
  const TraceKernel kernel =
      !by_rule ? tv->kernel
      : bvh->face_count >= kFetchBoundFaces
          ? k_fast_trace_v<false, kTraceWG, kSpreadRun, kDeepestLdsStack, false, 0, 32, 1, true, true>
      : bvh->face_count >= kXcdFaces
          ? k_fast_trace_v<false, kTraceWG, kSpreadRun, kDeepLdsStack, false, 0, kTraceDonateMin, 1, true, true>
      : bvh->face_count >= kApartFaces
          ? k_fast_trace_v<false, kTraceWG, kSpreadRun, kDeepLdsStack, false, 0, kTraceDonateMin, 1, false, true>
          : k_fast_trace_v<false, kTraceWG, kSpreadRun, kDeepLdsStack, false, 0, kTraceDonateMin>;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(n_rays, tv->wg)), dim3(tv->wg), 0, st, nodes,
                     static_cast<const float4*>(bvh->tris), bvh->face_count, o,
                     reinterpret_cast<const float4*>(directions), n_rays, faces_id, reinterpret_cast<float2*>(coords),
                     depths, det_eps_of(options), (unsigned long long*)nullptr, (const uint32_t*)order,
                     trace_flags_of(options));
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}
