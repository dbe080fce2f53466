// Closest-hit traversal of the reference tree layout (bvnode, 32 B) with the
// reference arithmetic (CUDA_raytraceMeshTree.cu), for gfx950:
//   k_tri_records   the call's triangle records, and bounds of each 16 and 64
//                   faces (rk_face_bounds.h): every leaf test below skips the
//                   groups of faces its ray misses
//   k_trace_ray     per-ray DFS (kernel_raytraceMeshTree, :111-219), one lane
//                   per ray for the nodes; a leaf's faces tested by its lane,
//                   or by the whole wave when few lanes hold a leaf; stack in
//                   LDS and scratch
//   k_trace_packet  the 16x12 packet traversal (kernel_raytraceMeshTreePacket,
//                   :222-377), one 192-thread workgroup (3 waves) per tile,
//                   block-uniform stack in LDS, one barrier vote per node
//   k_units_cut, k_unit_walk, k_units_merge, k_packet_commit
//                   rays that pass every box test, and the packets that hold
//                   one: their walks cut into subtrees, walked for groups of
//                   64 rays and merged in walk order
//   k_trace_ray_wave  other rays past a face budget: the same walk, one wave
//                   per ray, leaves tested by the whole wave
//   k_trace_packet_split  other packets past a face budget: the same walk with
//                   five threads per ray, each testing a fifth of every leaf
// The results are bit-identical to the reference's.
// Built with -ffp-contract=off, so the triangle and box tests are the same
// float operations in the same order as the reference source.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "rk_device.h"
#include "rk_face_bounds.h"

namespace {

constexpr float kEps = 0.000001f;  // CUDA_raytraceMeshTree.cu:36
constexpr float kUMargin = 0.001f;
#ifndef RK_REF_U_PRETEST
#define RK_REF_U_PRETEST 1
#endif

// intersectTriRay, CUDA_raytraceMeshTree.cu:57-89.
__device__ __forceinline__ bool tri_ray(float4 orig, float4 dir, float4 v0, float4 e1, float4 e2, float& t, float& u,
                                        float& v) {
  float4 pvec = rk::cross4(dir, e2);
  float det = rk::dot4(e1, pvec);
  if (det > -kEps && det < kEps) return false;
  float4 tvec = rk::sub4(orig, v0);
  const float un = rk::dot4(tvec, pvec);
  // Most faces fail on u. Estimated with the hardware reciprocal (within
  // 2^-21 of 1/det), a u below -kUMargin or above 1 + kUMargin means a u
  // computed with the correctly rounded 1/det is outside [0, 1] too (with the
  // same sign, also past the float range); NaN and every other case go on to
  // the exact division. The result is the reference's in every case.
#if RK_REF_U_PRETEST
  const float ua = un * __builtin_amdgcn_rcpf(det);
  if (ua < -kUMargin || ua > 1.0f + kUMargin) return false;
#endif
  float inv_det = 1.0f / det;
  u = un * inv_det;
  if (u < 0.0f || u > 1.0f) return false;
  float4 qvec = rk::cross4(tvec, e1);
  v = rk::dot4(dir, qvec) * inv_det;
  if (v < 0.0f || u + v > 1.0f) return false;
  t = rk::dot4(e2, qvec) * inv_det;
  return t >= 0.0f;
}

// intersectBoxRay, CUDA_raytraceMeshTree.cu:91-105.
__device__ __forceinline__ bool box_ray(float4 bmin, float4 bmax, float4 orig, float4 invdir, float& t) {
  float4 v1 = rk::mul4(rk::sub4(bmin, orig), invdir);
  float4 v2 = rk::mul4(rk::sub4(bmax, orig), invdir);
  float4 vmin = rk::min4(v1, v2);
  float4 vmax = rk::max4(v1, v2);
  float tmin = rk::fmx(vmin.z, rk::fmx(vmin.x, vmin.y));
  float tmax = rk::fmn(vmax.z, rk::fmn(vmax.x, vmax.y));
  t = tmin;
  return (tmax >= tmin) && (tmax >= 0.0f);
}

// invdir = normalize(1/dir), :128, with normalize read as v * (1.0f / sqrtf(dot(v, v))).
__device__ __forceinline__ float4 invdir_of(float4 dir) {
  float4 v = make_float4(1.0f / dir.x, 1.0f / dir.y, 1.0f / dir.z, 0.0f);
  float inv_len = 1.0f / __builtin_sqrtf(rk::dot4(v, v));
  return rk::muls4(v, inv_len);
}

// Whether box_ray passes every box for this invdir while t < depth allows:
// a direction component of 0 makes 1/dir infinite, the normalisation factor
// 0 and that component NaN; the other components are then +-0, and
// box_ray's tmin and tmax are both 0.
__device__ __forceinline__ bool crosses_every_box(float4 invdir) {
  return __builtin_isnan(invdir.x) || __builtin_isnan(invdir.y) || __builtin_isnan(invdir.z);
}

__device__ __forceinline__ void tri_setup(const uint4* __restrict__ faces, const float4* __restrict__ verts, uint32_t f,
                                          float4& v0, float4& e1, float4& e2) {
  uint4 face = faces[f];
  v0 = verts[face.x];
  e1 = rk::sub4(verts[face.y], v0);
  e2 = rk::sub4(verts[face.z], v0);
  v0.w = 0.0f;
  e1.w = 0.0f;
  e2.w = 0.0f;
}

// A face's tri_setup terms, v0, e1 = v1 - v0 and e2 = v2 - v0 (w 0),
// precomputed per call in face order (nine floats, 36 B per face): one
// contiguous load per face test instead of the face's indices, then its
// vertices. And the bound of each kFaceGroup faces (rk_face_bounds.h), 2 B per
// face, and of each wave's 64: reduced by shuffles.
constexpr size_t kRecFloats = 9;
constexpr uint32_t kGroup = rk::kFaceGroup;
constexpr uint32_t kSuper = 64 / kGroup;
static_assert(kGroup == 16, "a group is a quarter of a wave");
__global__ __launch_bounds__(256) void k_tri_records(const uint4* __restrict__ faces,
                                                     const float4* __restrict__ verts, uint32_t face_count,
                                                     float* __restrict__ tris, rk::FaceBound* __restrict__ bounds,
                                                     rk::FaceBound* __restrict__ supers) {
  const uint32_t f = blockIdx.x * 256 + threadIdx.x;
  const bool in = f < face_count;
  float lo[3], hi[3], e2m = 0.0f, nan = 0.0f;
  for (int q = 0; q < 3; ++q) { lo[q] = RK_HUGE; hi[q] = -RK_HUGE; }
  if (in) {
    const uint4 face = faces[f];
    const float4 a = verts[face.x], b = verts[face.y], c = verts[face.z];
    const float4 e1 = rk::sub4(b, a), e2 = rk::sub4(c, a);
    float3* r = reinterpret_cast<float3*>(tris + kRecFloats * (size_t)f);
    r[0] = make_float3(a.x, a.y, a.z);
    r[1] = make_float3(e1.x, e1.y, e1.z);
    r[2] = make_float3(e2.x, e2.y, e2.z);
    lo[0] = fminf(fminf(a.x, b.x), c.x); hi[0] = fmaxf(fmaxf(a.x, b.x), c.x);
    lo[1] = fminf(fminf(a.y, b.y), c.y); hi[1] = fmaxf(fmaxf(a.y, b.y), c.y);
    lo[2] = fminf(fminf(a.z, b.z), c.z); hi[2] = fmaxf(fmaxf(a.z, b.z), c.z);
    const float l1 = e1.x * e1.x + e1.y * e1.y + e1.z * e1.z, l2 = e2.x * e2.x + e2.y * e2.y + e2.z * e2.z;
    e2m = fmaxf(l1, l2);
    nan = l1 + l2;  // NaN or infinite when a vertex is (fminf and fmaxf drop NaN)
  }
  // (lane 0 of a group or wave with any face holds one: faces fill them from the front)
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    if (off == (int)kGroup && in && f % kGroup == 0)
      bounds[f / kGroup] = rk::face_bound(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], nan == nan ? 1.00001f * e2m : nan);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lo[q] = fminf(lo[q], __shfl_xor(lo[q], off, 64));
      hi[q] = fmaxf(hi[q], __shfl_xor(hi[q], off, 64));
    }
    e2m = fmaxf(e2m, __shfl_xor(e2m, off, 64));
    nan += __shfl_xor(nan, off, 64);
  }
  if (in && f % 64 == 0)
    supers[f / 64] = rk::face_bound(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], nan == nan ? 1.00001f * e2m : nan);
}

// One of a record's three vectors, w 0 as tri_setup leaves it.
__device__ __forceinline__ float4 rec_vec(const float* __restrict__ r) {
  const float3 v = *reinterpret_cast<const float3*>(r);
  return make_float4(v.x, v.y, v.z, 0.0f);
}

// The call's faces: the mesh, and the records and bounds k_tri_records wrote
// (both NULL when there was no memory for them).
struct RefMesh {
  const uint4* faces;
  const float4* verts;
  const float* tris;
  const rk::FaceBound* bounds;  // per kGroup faces
  const rk::FaceBound* supers;  // per kSuper groups (a wave's 64 faces)
};

// tri_setup from the records when the call has them, else from the mesh.
__device__ __forceinline__ void tri_get(const RefMesh& m, uint32_t f, float4& v0, float4& e1, float4& e2) {
  if (m.tris) {
    const float* r = m.tris + kRecFloats * (size_t)f;
    v0 = rec_vec(r);
    e1 = rec_vec(r + 3);
    e2 = rec_vec(r + 6);
  } else {
    tri_setup(m.faces, m.verts, f, v0, e1, e2);
  }
}

__device__ __forceinline__ rk::CullRay cull_ray4(float4 o, float4 d) {
  return rk::cull_ray(o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w);
}

#ifndef RK_REF_BOUND_BATCH
#define RK_REF_BOUND_BATCH 4
#endif
constexpr uint32_t kBoundBatch = RK_REF_BOUND_BATCH;
// Which of the groups g0 .. g0 + ng - 1 (ng <= 32) may hold a face the ray's
// part [0, depth] hits: bit j for group g0 + j. Every group without bounds.
__device__ __forceinline__ uint32_t groups_near(const rk::FaceBound* __restrict__ bounds, uint32_t g0, uint32_t ng,
                                                float4 o, float4 d, const rk::CullRay& cr, float depth) {
  if (!bounds) return ng >= 32u ? 0xFFFFFFFFu : (1u << ng) - 1u;
  uint32_t mask = 0u;
  for (uint32_t j0 = 0; j0 < ng; j0 += kBoundBatch) {  // their loads in flight together
    rk::FaceBound b[kBoundBatch];
#pragma unroll
    for (uint32_t j = 0; j < kBoundBatch; ++j) b[j] = bounds[g0 + min(j0 + j, ng - 1u)];
#pragma unroll
    for (uint32_t j = 0; j < kBoundBatch; ++j)
      if (j0 + j < ng && !rk::bound_missed(b[j], o.x, o.y, o.z, d.x, d.y, d.z, cr, depth)) mask |= 1u << (j0 + j);
  }
  return mask;
}

// One lane's pass over faces [first, first + cnt) in face order, keeping a hit
// when t < depth: (depth, fid, uv) as a sequential pass over all of them ends.
// Faces of groups the ray misses are skipped; the lanes of a wave step through
// the faces left to each, so the pass lasts as long as the most any lane has.
// On the 1920x1080 frame of the 1M-face terrain (leaves of 155 faces, 10
// groups, of which a ray meets one or two) the per-ray first pass takes 1.48 ms
// with the groups skipped and 2.97 without, the packets' 0.66 and 1.58 ms. It
// is bound by the latency of its loads: 4 faces and 4 bounds in flight per
// lane against 2 and 2, 2.02 against 2.13 ms per frame (1 face: 2.31; 8: 2.11).
#ifndef RK_REF_LEAF_BATCH
#define RK_REF_LEAF_BATCH 4
#endif
constexpr uint32_t kLeafBatch = RK_REF_LEAF_BATCH;
__device__ __forceinline__ void lane_leaf(const RefMesh& mesh, uint32_t first, uint32_t cnt, float4 o, float4 d,
                                          const rk::CullRay& cr, float& depth, uint32_t& fid, float2& coord) {
  if (cnt == 0u) return;
  const uint32_t end = first + cnt, g_end = (end - 1u) / kGroup + 1u;
  for (uint32_t g0 = first / kGroup; g0 < g_end; g0 += 32u) {
    uint32_t mask = groups_near(mesh.bounds, g0, min(32u, g_end - g0), o, d, cr, depth);
    uint32_t f = 0u, stop = 0u;
    for (;;) {
      if (f >= stop) {
        if (mask == 0u) break;
        const uint32_t g = (g0 + (uint32_t)__builtin_ctz(mask)) * kGroup;
        mask &= mask - 1u;
        f = max(first, g);
        stop = g + min(end - g, kGroup);
      }
      float4 v0[kLeafBatch], e1[kLeafBatch], e2[kLeafBatch];
#pragma unroll
      for (uint32_t b = 0; b < kLeafBatch; ++b) tri_get(mesh, min(f + b, stop - 1u), v0[b], e1[b], e2[b]);
#pragma unroll
      for (uint32_t b = 0; b < kLeafBatch; ++b) {
        float t, u, v;
        if (f + b < stop && tri_ray(o, d, v0[b], e1[b], e2[b], t, u, v)) {
          if (t < depth) { fid = f + b; coord = make_float2(u, v); depth = t; }
        }
      }
      f += kLeafBatch;
    }
  }
}

// The same pass without the bounds, kB faces in flight: for leaves of few faces.
// Finding the groups of faces a ray is near costs one more round trip to memory per
// leaf, and round trips are what a frame of few waves is made of.
template <uint32_t kB>
__device__ __forceinline__ void plain_leaf(const RefMesh& mesh, uint32_t f, uint32_t end, float4 o, float4 d,
                                           float& depth, uint32_t& fid, float2& coord) {
  for (; f < end; f += kB) {
    float4 v0[kB], e1[kB], e2[kB];
#pragma unroll
    for (uint32_t b = 0; b < kB; ++b) tri_get(mesh, min(f + b, end - 1u), v0[b], e1[b], e2[b]);
#pragma unroll
    for (uint32_t b = 0; b < kB; ++b) {
      float t, u, v;
      if (f + b < end && tri_ray(o, d, v0[b], e1[b], e2[b], t, u, v)) {
        if (t < depth) { fid = f + b; coord = make_float2(u, v); depth = t; }
      }
    }
  }
}

struct NodeRegs { uint32_t w0, w1; float4 bmin, bmax; };

__device__ __forceinline__ NodeRegs load_node(const rk::Node* __restrict__ nodes, uint32_t id) {
  const uint4* p = reinterpret_cast<const uint4*>(nodes + id);
  uint4 a = p[0], b = p[1];
  NodeRegs r;
  r.w0 = a.x; r.w1 = a.y;
  r.bmin = make_float4(__uint_as_float(a.z), __uint_as_float(a.w), __uint_as_float(b.x), 0.0f);
  r.bmax = make_float4(__uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w), 0.0f);
  return r;
}

// getChildren, CUDANode.h:113-127: a negative direction on the split axis visits child_id+1 first.
__device__ __forceinline__ void children_order(uint32_t w0, uint32_t w1, float4 dir, uint32_t& nearc, uint32_t& farc) {
  uint32_t ax = rk::node_axis(w0);
  bool neg = ax == 0 ? dir.x < 0.0f : (ax == 1 ? dir.y < 0.0f : dir.z < 0.0f);
  nearc = neg ? w1 + 1 : w1;
  farc = neg ? w1 : w1 + 1;
}

constexpr int kStack = 96;  // STACK_SIZE, :45
#ifndef RK_REF_LDS_STACK
#define RK_REF_LDS_STACK 32
#endif
constexpr int kLdsStack = RK_REF_LDS_STACK;  // entries per lane in LDS (8 KB per wave); the rest in scratch

__device__ __forceinline__ uint32_t readlane_u32(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ float readlane_f32(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ float4 readlane_f4(float4 v, int l) {
  return make_float4(readlane_f32(v.x, l), readlane_f32(v.y, l), readlane_f32(v.z, l), readlane_f32(v.w, l));
}

// The hand-off list of the per-ray traversal: word 0 counts the rays handed
// off, the ray indices start at word kHandoffHead.
constexpr uint32_t kHandoffHead = 64;
constexpr uint32_t kHandoffCap = 1u << 16;  // rays per call (256 KB)
constexpr uint32_t kRayWaveGrid = 8192;  // one-wave workgroups walking the other rays handed off

struct LeafBest { float t, u, v; uint32_t k; bool found; };

// The whole wave tests faces [first, first + cnt) against one ray (o, d, dep:
// the same in every lane) and returns the first face of smallest t < dep, the
// face a sequential pass keeping hits with t < depth would end on: its depth
// after such a pass is the smallest t below dep, and a later face with the
// same t fails t < depth. Each lane tests one group's bound, then the faces of
// four groups the ray may hit at a time, one face per lane, so that lane
// order is face order: the lowest lane holding the wave's smallest t has the
// first such face. The next four compare with that t. A leaf of at most 'plain'
// (<= 64) faces is tested without the bounds, in one round trip.
__device__ __forceinline__ LeafBest wave_leaf(const RefMesh& mesh, float4 o, float4 d, const rk::CullRay& cr,
                                              uint32_t first, uint32_t cnt, float dep, uint32_t plain) {
  const uint32_t lane = threadIdx.x & 63u, quarter = lane / kGroup;
  LeafBest r;
  r.t = dep;
  r.u = 0.0f;
  r.v = 0.0f;
  r.k = 0;
  r.found = false;
  const float inf = __int_as_float(0x7f800000);
  auto test = [&](bool has, uint32_t f) {  // a face per lane
    float bt = inf, bu = 0.0f, bv = 0.0f;
    bool any = false;
    if (has) {
      float4 v0, e1, e2;
      tri_get(mesh, f, v0, e1, e2);
      float t, u, v;
      if (tri_ray(o, d, v0, e1, e2, t, u, v) && t < r.t) {
        bt = t;  // t < dep <= FLT_MAX or +inf: t is finite, below the sentinel
        bu = u;
        bv = v;
        any = true;
      }
    }
    if (__ballot(any) == 0ull) return;
    float mn = bt;
    for (int off = 32; off > 0; off >>= 1) mn = fminf(mn, __shfl_xor(mn, off, 64));
    const int w = __builtin_ctzll(__ballot(any && bt == mn));
    r.t = __shfl(bt, w, 64);  // the winner's own bits (bt == mn holds for -0 against +0 too)
    r.u = __shfl(bu, w, 64);
    r.v = __shfl(bv, w, 64);
    r.k = (uint32_t)__shfl((int)(f - first), w, 64);
    r.found = true;
  };
  if (cnt <= plain) {
    test(lane < cnt, first + lane);
    return r;
  }
  const uint32_t end = first + cnt, g_end = (end - 1u) / kGroup + 1u;
  for (uint32_t g0 = first / kGroup; g0 < g_end; g0 += 64u) {
    bool near = lane < g_end - g0;
    if (near && mesh.bounds)
      near = !rk::bound_missed(mesh.bounds[g0 + lane], o.x, o.y, o.z, d.x, d.y, d.z, cr, r.t);
    uint64_t mask = __ballot(near);
    while (mask != 0ull) {
      uint32_t g = 0u;  // this quarter's group
      bool has = false;
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        if (mask != 0ull) {
          if (quarter == q) {
            g = (uint32_t)__builtin_ctzll(mask);
            has = true;
          }
          mask &= mask - 1ull;
        }
      }
      const uint32_t f = (g0 + g) * kGroup + lane % kGroup;
      test(has && f >= first && f < end, f);
    }
  }
  return r;
}

// Walks split by subtree: rays that pass every box test (crosses_every_box).
// The walk of such a ray visits every node below one that passes its box
// test, in an order fixed by its direction's octant, as long as its depth
// stays above 0 (its box tests give t = +-0); at depth 0 no later face can be
// kept (t < 0 never holds). So the subtrees at tree level kUnitLevel (and the
// leaves above it), each walked on its own from the ray's starting depth,
// give the walk's result when merged in walk order, first smallest t winning.
// A packet holding such a ray (the forcing ray) visits the same nodes in the
// order its first ray gives, whatever its other rays hold, as long as the
// forcing ray's depth stays above 0: its rays' walks are split the same way.
//
// k_units_cut finds the subtrees' roots once per octant, on the assumption
// that every box above the cut is passed; k_unit_walk walks one subtree for a
// group of 64 rays (rays of one octant, or a third of a packet), checking the
// boxes, and lists each ray's best hit in it; k_units_merge and
// k_packet_commit take each ray's first smallest t. What does not fit the
// assumption (a box failed, a stack overflow, a child out of range, more pops
// than the visit limit, the hit list full) is walked again as the reference
// does: a ray by one wave, a packet by k_trace_packet_split.
//
// Nearly every face of the tree is far from any one ray, so a walk is a scan
// of bounds, 64 faces at a time. On the 1920x1080 frame of the 1M-face terrain
// (1,949 such rays; 149 packets holding one; depth-12 LBVH, 155 faces per
// leaf) the subtree walks take 0.24 ms for the rays and 1.36 ms for the
// packets. With every face tested by every ray they took 2.76 ms, and the
// packets 37.9 ms in parts of 16 rays that each walked the whole tree. Cut
// level 7: 2.20 ms per per-ray frame against 2.02, packets the same.
#ifndef RK_REF_UNIT_LEVEL
#define RK_REF_UNIT_LEVEL 8
#endif
constexpr int kUnitLevel = RK_REF_UNIT_LEVEL;
constexpr uint32_t kUnits = 1u << kUnitLevel;  // subtrees at most: the cut has <= 2^kUnitLevel nodes
#ifndef RK_REF_CROSS_CAP
#define RK_REF_CROSS_CAP 4096
#endif
constexpr uint32_t kCrossCap = RK_REF_CROSS_CAP;  // rays split per call
constexpr uint32_t kUnitGrid = 8192;              // one-wave workgroups walking the subtrees
constexpr uint32_t kNone = 0xffffffffu;

// The subtrees of each direction octant (bit 0: x < 0, 1: y, 2: z), in walk order.
struct UnitCut {
  uint32_t units[8];            // subtrees
  uint32_t tops[8];             // internal nodes above them
  uint32_t node[8][kUnits];     // each subtree's root
  uint32_t sp[8][kUnits];       // the reference's stack size after popping that root
  uint32_t top[8][kUnits];      // the internal nodes above
};

// A ray's best hit in one subtree; next: the ray's previous entry, or kNone.
struct UnitHit { float t, u, v; uint32_t face, unit, next; };

// The split walks' state in the hand-off buffer. A slot is a crossing ray's
// place in list, or a forced packet's ray (packet's place * kPT + ray).
struct UnitArgs {
  uint32_t* list;            // crossing rays: [cap] the rays, in hand-off order
  uint32_t* bucket;          // crossing rays: [8 * cap] the slots of each octant
  uint32_t* redo;            // crossing rays: [cap] the rays to walk again
  uint32_t* diverged;        // [cap] per crossing ray or forced packet: walk it again
  unsigned long long* pops;  // per group: pops of its subtree walks
  uint32_t* head;            // per slot: its last hit entry, or kNone
  UnitHit* hits;             // [hit_cap]
  UnitCut* cut;
  uint32_t cap, hit_cap;
};
// Words of the hand-off buffer's head: [0] handed off, [1] crossing rays, [2]
// forced packets, [3] hit entries, [4] crossing rays to walk again.
constexpr uint32_t kBucketHead = 8;  // [8 + o]: crossing rays of octant o
__device__ __forceinline__ uint32_t octant_of(float4 dir) {
  return (dir.x < 0.0f ? 1u : 0u) | (dir.y < 0.0f ? 2u : 0u) | (dir.z < 0.0f ? 4u : 0u);
}

// The per-ray traversal (kernel_raytraceMeshTree, :111-219), one lane per ray:
// pop a node, test its box against the depth so far, push the far child, then
// the near one; at a leaf, test its faces in order, keeping a hit only when
// t < depth. Each ray's result is bit-identical to the reference's.
//
// The lanes of a wave walk their nodes until each has reached a leaf or its
// end; then the leaves are tested, and the walk goes on. A frame's cost sits
// in a few rays that graze the scene and cross dozens of leaves of a few
// hundred faces each: on the 1920x1080 heightfield the waves that hold them
// ran alone for most of the frame (0.5 waves per CU on average). So when at
// most kCoopMax lanes hold a leaf, the whole wave tests each of those leaves
// in turn (wave_leaf): the same depth after every leaf as the reference's, and
// so the same later pops. When more lanes hold a leaf, each lane tests its own
// (lane_leaf). Both skip the groups of faces the ray misses.
//
// The stack keeps the reference's 96 entries and its overflow rule; the first
// kLdsStack entries of each lane live in LDS (entry e of lane x at
// e * 64 + x), deeper ones in scratch (trees of depth <= 31 need at most 33),
// so a CU holds 16 waves of this kernel instead of 6, as its 101 registers allow (20,
// with 7 spilled: no faster over 140 frames).
//
// A wave's rays are a tile of 16 x 4 pixels where that fills nearly all lanes
// (tiled_rays), else 64 in a row: neighbours in the picture walk the same nodes
// to the same leaves. The 1920x1080 heightfield frame: 2.02 -> 1.82 ms with 16 x 4 (8
// x 8: 1.96, 32 x 2: 1.85, 4 x 16: 1.93); at tree depths 20 and 31, 2.55 -> 2.70 and
// 3.50 -> 3.63, from another side 2.41 -> 2.25.
//
// Not below kTileRays, a wave per SIMD: such a frame takes as long as its longest
// wave, and where the mesh fills a small part of the picture tiles gather the rays
// that reach a leaf into few waves (95x53 frame of a 2k-face heightfield from afar 223
// us tiled, 154 in rows; 111x62 of 90,000 scattered faces 676 and 485).
//
// Leaves of at most 16 faces go without the bounds (320-face sphere, 253x142: 165 ->
// 147 us), and in frames in rows, which are made of round trips to memory, leaves of at
// most 64 where the whole wave tests one. Large frames of many scattered faces
// would gain from bounds there too (68,000 faces, 1902x1902: 13.3 ms, 15.0 so), but
// close views of few large ones would be slower than with every face tested (345
// faces, 1548x1548: 1.56 ms, 1.36 so, 1.43 then).
//
// Over 110 random frames of up to 400x400, 260 of 200x112 to 1920x1920, near and far
// views, and 200 of the terrains' and spheres' usual ones: 1.24, 1.43 and 1.74 times as
// fast as with every face tested, one of them slower (0.87, 800 faces from afar). With
// tiles and bounds for all: 1.14, 1.37 and 1.66, sixty slower, down to 0.63.
constexpr uint32_t kTileW = 16, kTileH = 64 / kTileW;
constexpr uint64_t kTileRays = 1u << 16;
inline bool tiled_rays(uint32_t width, uint32_t height) {  // at most an eighth of the lanes without a ray
  const uint64_t n = (uint64_t)width * height;
  const uint64_t tiles = ((uint64_t)width + kTileW - 1) / kTileW * (((uint64_t)height + kTileH - 1) / kTileH);
  return n >= kTileRays && 64 * tiles <= n + n / 8;
}
template <int kCoopMax>
__global__ __launch_bounds__(64) void k_trace_ray(const rk::Node* __restrict__ nodes,
                                                  RefMesh mesh,
                                                  const float4* __restrict__ origins,
                                                  const float4* __restrict__ dirs, uint32_t n_rays,
                                                  uint32_t width, uint32_t height, uint32_t tiles_x,
                                                  uint32_t node_count, uint32_t face_count,
                                                  uint32_t* __restrict__ faces_id,
                                                  float2* __restrict__ coords, float* __restrict__ depths,
                                                  uint32_t* __restrict__ handoff, uint32_t handoff_cap,
                                                  uint32_t handoff_faces, UnitArgs ua) {
  __shared__ uint32_t s_stack[kLdsStack * 64];
  const int lane = (int)threadIdx.x;
  uint32_t l = blockIdx.x * 64 + (uint32_t)lane;
  bool has_ray = l < n_rays;
  if (tiles_x != 0u) {  // 0: in a row
    const uint32_t x = blockIdx.x % tiles_x * kTileW + (uint32_t)lane % kTileW;
    const uint32_t y = blockIdx.x / tiles_x * kTileH + (uint32_t)lane / kTileW;
    l = y * width + x;
    has_ray = x < width && y < height;
  }
  const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float4 orig = has_ray ? origins[l] : zero4, dir = has_ray ? dirs[l] : zero4;
  const float4 invdir = has_ray ? invdir_of(dir) : zero4;
  const rk::CullRay cr = cull_ray4(orig, dir);
  float depth = has_ray ? depths[l] : 0.0f;
  uint32_t fid = has_ray ? faces_id[l] : 0u;
  float2 coord = has_ray ? coords[l] : make_float2(0.0f, 0.0f);
  uint32_t spill[kStack - kLdsStack];
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  lds_u32* my_lds = (lds_u32*)(s_stack + lane);
  int sp = 0;
  if (has_ray) {
    my_lds[0] = 0u;
    sp = 1;
  }
  bool active = has_ray;
  bool may_hand_off = handoff_cap != 0u, handed_off = false;
  uint32_t tested = 0;  // faces of the leaves reached, while may_hand_off
  // A direction with a component of 0 leaves a NaN in invdir: every box test
  // then passes (at t = 0, while depth > 0) and the ray walks the whole tree,
  // so it goes to the split at once (else to the second pass at its first leaf).
  const bool crossing = has_ray && crosses_every_box(invdir);
  const uint32_t limit = crossing ? 0u : handoff_faces;
  if (crossing && may_hand_off && ua.cap != 0u) {
    const uint32_t slot = atomicAdd(handoff + 1, 1u);
    if (slot < ua.cap) {
      const uint32_t o = octant_of(dir);
      ua.list[slot] = l;
      ua.diverged[slot] = 0u;
      ua.head[slot] = kNone;
      ua.bucket[o * ua.cap + atomicAdd(handoff + kBucketHead + o, 1u)] = slot;  // at most cap rays in all
      handed_off = true;
      active = false;
    }
  }
  uint32_t visits = 0;
  const uint32_t max_visits = 2 * node_count + 2;
  for (;;) {
    // each lane walks on to its next leaf, or to its end
    bool at_leaf = false;
    uint32_t leaf_first = 0, leaf_cnt = 0;
    while (active && !at_leaf) {
      if (sp == 0 || ++visits > max_visits) {
        active = false;
        break;
      }
      --sp;
      const uint32_t nid = sp < kLdsStack ? my_lds[sp * 64] : spill[sp - kLdsStack];
      if (nid >= node_count) {  // never taken for a tree built by this library
        active = false;
        break;
      }
      const NodeRegs nd = load_node(nodes, nid);
      if (rk::node_is_leaf(nd.w0)) {
        leaf_first = nd.w1;
        leaf_cnt = leaf_first < face_count ? min(rk::leaf_count(nd.w0), face_count - leaf_first) : 0u;
        if (may_hand_off) {
          if (leaf_cnt > limit - tested) {
            may_hand_off = false;
            const uint32_t slot = atomicAdd(handoff, 1u);
            if (slot < handoff_cap) {
              handoff[kHandoffHead + slot] = l;
              handed_off = true;
              active = false;
              break;
            }
          } else {
            tested += leaf_cnt;
          }
        }
        at_leaf = true;
      } else {
        float t;
        if (box_ray(nd.bmin, nd.bmax, orig, invdir, t) && t < depth) {
          uint32_t nearc, farc;
          children_order(nd.w0, nd.w1, dir, nearc, farc);
          if (sp + 2 > kStack) {  // depth > 94: cannot occur for trees of depth <= 94
            active = false;
            break;
          }
          if (sp < kLdsStack) my_lds[sp * 64] = farc;
          else spill[sp - kLdsStack] = farc;
          ++sp;
          if (sp < kLdsStack) my_lds[sp * 64] = nearc;
          else spill[sp - kLdsStack] = nearc;
          ++sp;
        }
      }
    }
    uint64_t pending = __ballot(at_leaf);
    if (pending == 0ull) break;  // every lane is done
    if (__popcll(pending) > kCoopMax) {
      // each lane its own leaf, in face order
      const bool plain = __ballot(at_leaf && leaf_cnt > kGroup) == 0ull;
      if (at_leaf) {
        if (plain) plain_leaf<kLeafBatch>(mesh, leaf_first, leaf_first + leaf_cnt, orig, dir, depth, fid, coord);
        else lane_leaf(mesh, leaf_first, leaf_cnt, orig, dir, cr, depth, fid, coord);
      }
    } else {
      // the whole wave on each pending leaf in turn
      while (pending != 0ull) {
        const int L = __builtin_ctzll(pending);
        pending &= pending - 1;
        const uint32_t first = readlane_u32(leaf_first, L);
        const float4 oL = readlane_f4(orig, L), dL = readlane_f4(dir, L);
        const LeafBest b = wave_leaf(mesh, oL, dL, rk::CullRay{readlane_f32(cr.dl, L), readlane_f32(cr.d2, L)},
                                     first, readlane_u32(leaf_cnt, L), readlane_f32(depth, L),
                                     tiles_x != 0u ? kGroup : 64u);
        if (lane == L && b.found) {
          depth = b.t;
          fid = first + b.k;
          coord = make_float2(b.u, b.v);
        }
      }
    }
  }
  if (has_ray && !handed_off) {
    faces_id[l] = fid;
    coords[l] = coord;
    depths[l] = depth;
  }
}

// The cut: one workgroup per octant expands the tree level by level, in walk
// order, down to kUnitLevel; a leaf or a child out of range ends where it is.
// The reference's stack holds, after it pops a node, one far child for every
// near step on the path to it. The workgroups after the first eight clear the
// head's counters and the groups' pops.
__global__ __launch_bounds__(256) void k_units_cut(const rk::Node* __restrict__ nodes, uint32_t node_count,
                                                   UnitCut* __restrict__ cut, uint32_t* __restrict__ handoff,
                                                   unsigned long long* __restrict__ pops, uint32_t groups) {
  static_assert(kUnits <= 256, "one thread per subtree");
  __shared__ uint32_t s_node[kUnits], s_sp[kUnits], s_wave[4];
  constexpr uint32_t kDone = 0x80000000u;
  if (blockIdx.x >= 8u) {
    const uint32_t i = (blockIdx.x - 8u) * 256 + threadIdx.x;
    if (i < kHandoffHead) handoff[i] = 0u;
    if (i < groups) pops[i] = 0ull;
    return;
  }
  const uint32_t o = blockIdx.x, t = threadIdx.x, lane = t & 63u, wv = t >> 6;
  uint32_t n = 1, tops = 0;
  if (t == 0) {
    s_node[0] = 0u;
    s_sp[0] = 0u;
  }
  __syncthreads();
  for (int level = 0; level < kUnitLevel; ++level) {
    const bool in = t < n;
    const uint32_t nid = in ? s_node[t] : 0u;
    uint32_t sp = in ? s_sp[t] : 0u;
    bool expand = false;
    uint32_t w0 = 0, w1 = 0;
    if (in && !(sp & kDone)) {
      if (nid < node_count) {
        w0 = nodes[nid].w0;
        w1 = nodes[nid].w1;
        expand = !rk::node_is_leaf(w0);
      }
      if (!expand) sp |= kDone;
    }
    const uint64_t em = __ballot(expand);
    if (lane == 0) s_wave[wv] = (uint32_t)__popcll(em);
    __syncthreads();  // also: every entry has been read
    uint32_t before = (uint32_t)__popcll(em & rk::lanemask_lt()), total = 0;
    for (uint32_t w = 0; w < 4; ++w) {
      if (w < wv) before += s_wave[w];
      total += s_wave[w];
    }
    if (in) {
      const uint32_t at = t + before;
      if (expand) {
        const uint32_t ax = rk::node_axis(w0);
        const bool neg = ax <= 1u ? ((o >> ax) & 1u) != 0u : (o & 4u) != 0u;  // children_order
        s_node[at] = neg ? w1 + 1u : w1;
        s_sp[at] = sp + 1u;
        s_node[at + 1] = neg ? w1 : w1 + 1u;
        s_sp[at + 1] = sp;
        cut->top[o][tops + before] = nid;
      } else {
        s_node[at] = nid;
        s_sp[at] = sp;
      }
    }
    n += total;
    tops += total;
    __syncthreads();
  }
  if (t < n) {
    cut->node[o][t] = s_node[t];
    cut->sp[o][t] = s_sp[t] & ~kDone;
  }
  if (t == 0) {
    cut->units[o] = n;
    cut->tops[o] = tops;
  }
}

// The walk of ray l by the whole wave with the reference's rules (the same
// pops, box tests, stack overflow and visit limits), each leaf tested by the
// whole wave (wave_leaf), from the depth, face and coordinates given, into them.
// The stack's entry e is lane e % 64 of st0 (e < 64) or st1.
__device__ __forceinline__ void wave_walk(uint32_t l, float& depth, uint32_t& fid, float2& coord,
                                          const rk::Node* __restrict__ nodes, RefMesh mesh,
                                          const float4* __restrict__ origins, const float4* __restrict__ dirs,
                                          uint32_t node_count, uint32_t face_count) {
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t max_visits = 2 * node_count + 2;
  const float4 orig = origins[l], dir = dirs[l];
  const float4 invdir = invdir_of(dir);
  const rk::CullRay cr = cull_ray4(orig, dir);
  uint32_t st0 = 0u, st1 = 0u;  // the root
  int sp = 1;
  uint32_t visits = 0;
  while (sp > 0 && ++visits <= max_visits) {
    --sp;
    const uint32_t nid = readlane_u32(sp < 64 ? st0 : st1, sp & 63);
    if (nid >= node_count) break;  // never taken for a tree built by this library
    const NodeRegs nd = load_node(nodes, nid);
    if (rk::node_is_leaf(nd.w0)) {
      const uint32_t first = nd.w1;
      const uint32_t cnt = first < face_count ? min(rk::leaf_count(nd.w0), face_count - first) : 0u;
      const LeafBest b = wave_leaf(mesh, orig, dir, cr, first, cnt, depth, 64u);
      if (b.found) {
        depth = b.t;
        fid = first + b.k;
        coord = make_float2(b.u, b.v);
      }
    } else {
      float t;
      if (box_ray(nd.bmin, nd.bmax, orig, invdir, t) && t < depth) {
        uint32_t nearc, farc;
        children_order(nd.w0, nd.w1, dir, nearc, farc);
        if (sp + 2 > kStack) break;  // cannot occur for trees of depth <= 94
        if (lane == (sp & 63)) {
          if (sp < 64) st0 = farc;
          else st1 = farc;
        }
        ++sp;
        if (lane == (sp & 63)) {
          if (sp < 64) st0 = nearc;
          else st1 = nearc;
        }
        ++sp;
      }
    }
  }
}

// The second pass of the per-ray traversal: one wave per ray handed off (and
// per crossing ray whose split walk did not fit), its walk again from the root.
__global__ __launch_bounds__(64) void k_trace_ray_wave(const rk::Node* __restrict__ nodes,
                                                       RefMesh mesh,
                                                       const float4* __restrict__ origins,
                                                       const float4* __restrict__ dirs, uint32_t node_count,
                                                       uint32_t face_count, const uint32_t* __restrict__ handoff,
                                                       uint32_t handoff_cap, const uint32_t* __restrict__ redo,
                                                       uint32_t redo_cap, uint32_t* __restrict__ faces_id,
                                                       float2* __restrict__ coords, float* __restrict__ depths) {
  const uint32_t count = min(handoff[0], handoff_cap), again = min(handoff[4], redo_cap);
  for (uint32_t i = blockIdx.x; i < count + again; i += gridDim.x) {
    const uint32_t l = i < count ? handoff[kHandoffHead + i] : redo[i - count];
    float depth = depths[l];
    uint32_t fid = faces_id[l];
    float2 coord = coords[l];
    wave_walk(l, depth, fid, coord, nodes, mesh, origins, dirs, node_count, face_count);
    if (threadIdx.x == 0) {
      faces_id[l] = fid;
      coords[l] = coord;
      depths[l] = depth;
    }
  }
}

// Uniform data through the scalar cache: read-only for the whole kernel.
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ u32x8 load_uniform32(const void* p) {
  return *(const __attribute__((address_space(4))) u32x8*)(uintptr_t)p;
}
__device__ __forceinline__ NodeRegs load_node_uniform(const rk::Node* __restrict__ nodes, uint32_t id) {
  const u32x8 a = load_uniform32(nodes + __builtin_amdgcn_readfirstlane(id));
  NodeRegs r;
  r.w0 = a[0];
  r.w1 = a[1];
  r.bmin = make_float4(__uint_as_float(a[2]), __uint_as_float(a[3]), __uint_as_float(a[4]), 0.0f);
  r.bmax = make_float4(__uint_as_float(a[5]), __uint_as_float(a[6]), __uint_as_float(a[7]), 0.0f);
  return r;
}
__device__ __forceinline__ rk::FaceBound load_bound_uniform(const rk::FaceBound* __restrict__ p, uint32_t g) {
  const u32x8 a = load_uniform32(p + __builtin_amdgcn_readfirstlane(g));
  return rk::FaceBound{__uint_as_float(a[0]), __uint_as_float(a[1]), __uint_as_float(a[2]), __uint_as_float(a[3]),
                       __uint_as_float(a[4]), __uint_as_float(a[5]), __uint_as_float(a[6]), __uint_as_float(a[7])};
}

// Faces [first, first + cnt) against the wave's rays, one per lane (test: the
// lanes that have one), in face order, each lane keeping hits with t < its
// depth. A group's bound is tested by every lane; the faces of a group that
// some ray may hit are fetched one per lane and handed round by readlane.
__device__ __forceinline__ void group_leaf(const RefMesh& mesh, uint32_t first, uint32_t cnt, bool test, float4 o,
                                           float4 d, const rk::CullRay& cr, float& depth, uint32_t& fid,
                                           float2& coord) {
  if (cnt == 0u) return;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t end = first + cnt, g_end = (end - 1u) / kGroup + 1u;
  for (uint32_t s0 = first / kGroup; s0 < g_end;) {
    // up to four groups at a time: all of them are missed by every ray of the
    // wave when their common bound is
    const uint32_t s1 = min(g_end, (s0 / kSuper + 1u) * kSuper);
    bool near = test;
    if (mesh.supers) {
      const rk::FaceBound sb = load_bound_uniform(mesh.supers, s0 / kSuper);
      near = test && !rk::bound_missed(sb, o.x, o.y, o.z, d.x, d.y, d.z, cr, depth);
    }
    if (__ballot(near) != 0ull) {
      for (uint32_t g = s0; g < s1; ++g) {
        bool hit = near;
        if (mesh.bounds) {
          const rk::FaceBound gb = load_bound_uniform(mesh.bounds, g);
          hit = near && !rk::bound_missed(gb, o.x, o.y, o.z, d.x, d.y, d.z, cr, depth);
        }
        if (__ballot(hit) == 0ull) continue;
        const uint32_t f0 = max(first, g * kGroup), nf = g * kGroup + min(end - g * kGroup, kGroup) - f0;
        float4 v0, e1, e2;
        tri_get(mesh, f0 + min(lane, nf - 1u), v0, e1, e2);
        for (uint32_t q = 0; q < nf; ++q) {
          const float4 qv0 = make_float4(readlane_f32(v0.x, q), readlane_f32(v0.y, q), readlane_f32(v0.z, q), 0.0f);
          const float4 qe1 = make_float4(readlane_f32(e1.x, q), readlane_f32(e1.y, q), readlane_f32(e1.z, q), 0.0f);
          const float4 qe2 = make_float4(readlane_f32(e2.x, q), readlane_f32(e2.y, q), readlane_f32(e2.z, q), 0.0f);
          float t, u, v;
          if (hit && tri_ray(o, d, qv0, qe1, qe2, t, u, v)) {
            if (t < depth) { fid = f0 + q; coord = make_float2(u, v); depth = t; }
          }
        }
      }
    }
    s0 = s1;
  }
}

constexpr int kPW = 16, kPH = 12, kPT = kPW * kPH;  // PACKET_BLOCK_*, :47-49
constexpr int kPStack = 128;                       // PACKET_STACK_SIZE, :51
constexpr uint32_t kPGroups = kPT / 64;            // groups of a packet
// A packet's record: sp, visits, the forcing ray (the first ray of the
// packet that passes every box test, or kNone), its forced slot (or kNone;
// kDone once the forced walk's results are in the outputs), the stack.
constexpr uint32_t kPStateWords = kPStack + 4;
constexpr uint32_t kDone = 0xfffffffeu;

// The image and the packets' records, for k_unit_walk on forced packets.
struct PacketArgs {
  int width, height, packets_x;
  uint32_t handoff_cap;
  const uint32_t* forced;  // [cap] each forced packet's place in the hand-off list
};

// One wave per group of 64 rays and subtree, lane r on the group's ray r; the
// wave walks the subtree once, and every ray tests the leaves' faces in face
// order against its own depth, as the reference does.
//
// Crossing rays (kPacket false), groups of one octant: a node is visited when
// a ray still walking (not diverged, depth above 0) passes its box test; a ray
// still walking that fails a visited node's test is marked diverged.
// Packets: a node is visited when the forcing ray passes its box test, and
// the packet is marked diverged when it does not.
//
// The subtrees' boxes above the cut are checked by the first subtree's wave.
template <bool kPacket>
__global__ __launch_bounds__(64) void k_unit_walk(const rk::Node* __restrict__ nodes, RefMesh mesh,
                                                  const float4* __restrict__ origins, const float4* __restrict__ dirs,
                                                  const float* __restrict__ depths, uint32_t node_count,
                                                  uint32_t face_count, uint32_t* __restrict__ handoff, UnitArgs ua,
                                                  PacketArgs pa) {
  const int lane = (int)threadIdx.x;
  uint32_t bcount[8], groups = 0;
  if (kPacket) {
    groups = min(handoff[2], ua.cap) * kPGroups;
  } else {
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      bcount[o] = handoff[kBucketHead + o];
      groups += (bcount[o] + 63u) / 64u;
    }
  }
  const uint64_t jobs = (uint64_t)groups * kUnits;
  const uint32_t max_visits = 2 * node_count + 2;
  constexpr uint32_t kLimit = kPacket ? (uint32_t)kPStack : (uint32_t)kStack;
  for (uint64_t jj = blockIdx.x; jj < jobs; jj += gridDim.x) {
    // subtree k of every group before subtree k + 1 of any: the waves running
    // together walk the same part of the tree and share it in the L2
    const uint32_t k = (uint32_t)(jj / groups), g = (uint32_t)(jj % groups);
    uint32_t o = 0, slot = 0, l = 0, div = 0;  // octant, this lane's slot and ray, its mark
    bool has_ray = false;
    float4 borig, bdir, border;  // the ray whose boxes are tested, and the one that gives the order
    if (kPacket) {
      const uint32_t f = g / kPGroups, rslot = pa.forced[f];
      const uint32_t* rec = handoff + kHandoffHead + pa.handoff_cap + (size_t)rslot * kPStateWords;
      const uint32_t pk = handoff[kHandoffHead + rslot], R = rec[2];
      const int x0 = (int)(pk % (uint32_t)pa.packets_x) * kPW, y0 = (int)(pk / (uint32_t)pa.packets_x) * kPH;
      const int q = (int)(g % kPGroups) * 64 + lane, x = x0 + q % kPW, y = y0 + q / kPW;
      has_ray = x < pa.width && y < pa.height;
      l = has_ray ? (uint32_t)y * (uint32_t)pa.width + (uint32_t)x : 0u;
      slot = f * (uint32_t)kPT + (uint32_t)q;
      div = f;
      const uint32_t lr = (uint32_t)(y0 + (int)R / kPW) * (uint32_t)pa.width + (uint32_t)(x0 + (int)R % kPW);
      borig = origins[lr];
      bdir = dirs[lr];
      border = dirs[(uint32_t)y0 * (uint32_t)pa.width + (uint32_t)x0];
      o = octant_of(border);
    } else {
      uint32_t gg = g;
      while (gg >= (bcount[o] + 63u) / 64u) {
        gg -= (bcount[o] + 63u) / 64u;
        ++o;
      }
      has_ray = gg * 64u + (uint32_t)lane < bcount[o];
      slot = has_ray ? ua.bucket[o * ua.cap + gg * 64u + (uint32_t)lane] : 0u;
      l = has_ray ? ua.list[slot] : 0u;
      div = slot;
    }
    o = __builtin_amdgcn_readfirstlane(o);
    if (k >= ua.cut->units[o]) continue;
    const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 orig = has_ray ? origins[l] : zero4, dir = has_ray ? dirs[l] : zero4;
    if (!kPacket) {
      borig = orig;
      bdir = dir;
      border = readlane_f4(dir, 0);  // the octant's
    }
    const float4 binv = invdir_of(bdir);
    const rk::CullRay cr = cull_ray4(orig, dir);
    float depth = has_ray ? depths[l] : 0.0f;
    uint32_t fid = kNone;
    float2 coord = make_float2(0.0f, 0.0f);
    bool walking = has_ray, diverged = false;
    if (k == 0) {  // every box above the cut, at the starting depth
      const uint32_t tops = ua.cut->tops[o];
      for (uint32_t i = 0; i < tops; ++i) {
        const NodeRegs nd = load_node_uniform(nodes, ua.cut->top[o][i]);
        float t;
        if (!(box_ray(nd.bmin, nd.bmax, borig, binv, t) && (kPacket || t < depth))) diverged = true;
      }
      if (!kPacket && diverged) walking = false;
    }
    const uint32_t root = ua.cut->node[o][k], sp_base = ua.cut->sp[o][k];
    uint32_t st0 = lane == 0 ? root : 0u, st1 = 0u;
    int sp = 1;
    uint32_t visits = 0;
    while (sp > 0 && ++visits <= max_visits) {
      if (!kPacket && __ballot(walking && depth > 0.0f) == 0ull) break;  // every ray's result here is final
      --sp;
      const uint32_t nid = readlane_u32(sp < 64 ? st0 : st1, sp & 63);
      if (nid >= node_count) {  // never taken for a tree built by this library
        diverged = true;
        break;
      }
      const NodeRegs nd = load_node_uniform(nodes, nid);
      if (rk::node_is_leaf(nd.w0)) {
        const uint32_t first = nd.w1;
        const uint32_t cnt = first < face_count ? min(rk::leaf_count(nd.w0), face_count - first) : 0u;
        group_leaf(mesh, first, cnt, walking, orig, dir, cr, depth, fid, coord);
      } else {
        float t;
        bool pass = box_ray(nd.bmin, nd.bmax, borig, binv, t);
        bool visit;
        if (kPacket) {
          visit = __ballot(pass) != 0ull;  // the same in every lane
          if (!visit) diverged = true;
        } else {
          pass = pass && t < depth;
          const bool live = walking && depth > 0.0f;  // at depth 0 a ray's result is final
          visit = __ballot(live && pass) != 0ull;
          if (visit && live && !pass) {
            walking = false;
            diverged = true;
          }
        }
        if (visit) {
          uint32_t nearc, farc;
          children_order(nd.w0, nd.w1, border, nearc, farc);
          nearc = __builtin_amdgcn_readfirstlane(nearc);
          farc = __builtin_amdgcn_readfirstlane(farc);
          if ((uint32_t)sp + sp_base + 2u > kLimit) {  // cannot occur for trees of depth <= 94
            diverged = true;
            break;
          }
          if (lane == (sp & 63)) {
            if (sp < 64) st0 = farc;
            else st1 = farc;
          }
          ++sp;
          if (lane == (sp & 63)) {
            if (sp < 64) st0 = nearc;
            else st1 = nearc;
          }
          ++sp;
        }
      }
    }
    if (lane == 0) atomicAdd(ua.pops + g, (unsigned long long)visits);
    const bool hit = has_ray && fid != kNone;
    const uint64_t hm = __ballot(hit);
    if (hm != 0ull) {
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(handoff + 3, (uint32_t)__popcll(hm));
      base = __builtin_amdgcn_readfirstlane(base);
      if (hit) {
        const uint32_t e = base + (uint32_t)__popcll(hm & rk::lanemask_lt());
        if (e < ua.hit_cap) {
          UnitHit h;
          h.t = depth;
          h.u = coord.x;
          h.v = coord.y;
          h.face = fid;
          h.unit = k;
          h.next = atomicExch(ua.head + slot, e);
          ua.hits[e] = h;
        } else {
          diverged = true;
        }
      }
    }
    if (diverged && has_ray) ua.diverged[div] = 1u;
  }
}

// A slot's result: of its entries, the smallest t, the first subtree's of
// equal ones; false when it has none. Entries hold t below the starting depth.
__device__ __forceinline__ bool unit_best(const UnitArgs& ua, uint32_t slot, UnitHit& best) {
  bool any = false;
  uint32_t e = ua.head[slot];
  for (uint32_t n = 0; e != kNone && n < kUnits; ++n) {
    const UnitHit h = ua.hits[e];
    if (!any || h.t < best.t || (h.t == best.t && h.unit < best.unit)) best = h;
    any = true;
    e = h.next;
  }
  return any;
}

// The crossing rays' results, one lane per ray; a diverged ray, or one of a
// group whose pops pass the visit limit, goes on the list to walk again.
__global__ __launch_bounds__(64) void k_units_merge(uint32_t node_count, uint32_t* __restrict__ handoff, UnitArgs ua,
                                                    uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                    float* __restrict__ depths) {
  const uint64_t max_visits = 2 * node_count + 2;
  uint32_t group0 = 0;
  for (uint32_t o = 0; o < 8; ++o) {
    const uint32_t n = handoff[kBucketHead + o];
    for (uint32_t i = blockIdx.x * 64u + threadIdx.x; i < n; i += gridDim.x * 64u) {
      const uint32_t slot = ua.bucket[o * ua.cap + i], l = ua.list[slot];
      if (ua.diverged[slot] != 0u || ua.pops[group0 + i / 64u] + ua.cut->tops[o] > max_visits) {
        ua.redo[atomicAdd(handoff + 4, 1u)] = l;  // at most cap rays
        continue;
      }
      UnitHit h;
      if (unit_best(ua, slot, h)) {
        faces_id[l] = h.face;
        coords[l] = make_float2(h.u, h.v);
        depths[l] = h.t;
      }
    }
    group0 += (n + 63u) / 64u;
  }
}

#ifndef RK_REF_HANDOFF_FACES
#define RK_REF_HANDOFF_FACES 4096
#endif

#ifndef RK_REF_COOP_MAX
#define RK_REF_COOP_MAX 16
#endif

// One packet of the packet traversal (kernel_raytraceMeshTreePacket,
// :222-377): the block walks the tree once for its 16x12 rays, visiting a
// node when any of them passes its box test with t < its depth, in the order
// the first ray's direction gives; at a leaf every ray tests every face
// against its own depth, in face order. The block holds kS threads per ray:
// thread x serves ray x % 192, and with kS > 1 tests part x / 192 of each
// chunk of faces (consecutive faces, parts in face order). Each part keeps its
// first face of smallest t below the ray's depth at the chunk's start, and the
// first part with the smallest t wins: the face a sequential pass keeping hits
// with t < depth ends on, with the same depth after the chunk.
//
// A packet whose leaves pass handoff_faces faces (while handoff_cap != 0) is
// put on the hand-off list and left where it stands: its rays' hits so far in
// the outputs, and in its record of the state area its stack with the leaf
// back on top, sp and the visits before that leaf's pop (so that the second
// pass, given the record as resume, makes the same pops from there). Returns
// whether it was.
//
// Leaves of at most kPlainLeaf faces: the second pass tests a part's share of the
// faces without the bounds. A 93x52 frame of a small heightfield takes 1.50 ms with
// them, 1.09 so (loads of 2 faces in flight; 4: 1.15), the 1920x1080 frame the same
// with both. The first pass, which has many packets, does so for leaves of at most a
// group (a 1528x859 frame of the 1,280-face sphere: 218 -> 201 us; 24 and 48 faces: no
// gain), through the scalar cache, since every ray of the block tests the same faces:
// large frames of small meshes 3-5% faster than with a load per lane, 1714x964 of that
// sphere 244 -> 234 us (230 with every face tested); 4 faces in flight no better than 2
// (8: 8% slower). Close views of few large faces, where bounds skip little in larger
// leaves, stay slower than with every face tested from LDS: 1.82 against 1.56 ms at
// 1497x1497 of 1,126 scattered faces. Six waves per SIMD for five (2 faces at a time
// in larger leaves) make up for that, but cost large frames of terrains 5-8%.
constexpr uint32_t kPlainLeaf = 96, kPlainBatch = 2;
__device__ __forceinline__ void uniform_leaf(const RefMesh& mesh, uint32_t f, uint32_t end, float4 o, float4 d,
                                             float& depth, uint32_t& fid, float2& coord) {
  f = __builtin_amdgcn_readfirstlane(f);
  end = __builtin_amdgcn_readfirstlane(end);
  for (; f < end; f += kPlainBatch) {
    float4 v0[kPlainBatch], e1[kPlainBatch], e2[kPlainBatch];
#pragma unroll
    for (uint32_t b = 0; b < kPlainBatch; ++b) {
      typedef const __attribute__((address_space(4))) float uniform_float;
      uniform_float* r = (uniform_float*)(uintptr_t)(mesh.tris + kRecFloats * (size_t)min(f + b, end - 1u));
      v0[b] = make_float4(r[0], r[1], r[2], 0.0f);
      e1[b] = make_float4(r[3], r[4], r[5], 0.0f);
      e2[b] = make_float4(r[6], r[7], r[8], 0.0f);
    }
#pragma unroll
    for (uint32_t b = 0; b < kPlainBatch; ++b) {
      float t, u, v;
      if (f + b < end && tri_ray(o, d, v0[b], e1[b], e2[b], t, u, v)) {
        if (t < depth) { fid = f + b; coord = make_float2(u, v); depth = t; }
      }
    }
  }
}
template <int kS>
__device__ __forceinline__ bool trace_packet_job(
    const rk::Node* __restrict__ nodes, RefMesh mesh,
    const float4* __restrict__ origins, const float4* __restrict__ dirs, int width, int height, uint32_t node_count,
    uint32_t face_count, uint32_t* __restrict__ faces_id, float2* __restrict__ coords, float* __restrict__ depths,
    int bx, int by, uint32_t* __restrict__ handoff, uint32_t handoff_cap, uint32_t handoff_faces,
    uint32_t* __restrict__ state, uint32_t* __restrict__ forced_list, UnitArgs ua,
    const uint32_t* __restrict__ resume, uint32_t* s_stack, float4* s_dir0, uint32_t* s_slot, float* s_pt,
    float* s_pu, float* s_pv, uint32_t* s_pk) {
  const int ray = (int)threadIdx.x % kPT, part = (int)threadIdx.x / kPT;
  const int tx = ray % kPW, ty = ray / kPW;
  const int x = bx * kPW + tx, y = by * kPH + ty;
  const bool in_image = x < width && y < height;
  const uint32_t l = in_image ? (uint32_t)(y * width + x) : 0u;
  float4 orig = make_float4(0.f, 0.f, 0.f, 0.f), dir = orig, invdir = orig;
  float depth = 0.0f;
  uint32_t fid = 0;
  float2 coord = make_float2(0.f, 0.f);
  if (in_image) {
    orig = origins[l];
    dir = dirs[l];
    invdir = invdir_of(dir);
    depth = depths[l];
    fid = faces_id[l];
    coord = coords[l];
  }
  const rk::CullRay cr = cull_ray4(orig, dir);
  int sp = 1;
  uint32_t visits = 0;
  if (resume) {
    sp = (int)resume[0];
    visits = resume[1];
    for (int k = (int)threadIdx.x; k < sp; k += kPT * kS) s_stack[k] = resume[4 + k];
  }
  if (threadIdx.x == 0) {  // thread (0,0) of a block is always inside the image
    *s_dir0 = dir;
    if (!resume) s_stack[0] = 0;
  }
  bool may_hand_off = handoff_cap != 0u;
  // Hands the packet off where it stands (stack s_stack[0 .. sp), visits):
  // false when the list is full. f: its place among the forced packets.
  auto hand_off = [&](uint32_t forcer) {
    __syncthreads();  // s_slot and s_stack are settled
    if (threadIdx.x == 0) {
      const uint32_t slot = atomicAdd(handoff, 1u);
      if (slot < handoff_cap) {
        handoff[kHandoffHead + slot] = (uint32_t)by * gridDim.x + (uint32_t)bx;
        uint32_t f = kNone;
        if (forcer != kNone) {
          f = atomicAdd(handoff + 2, 1u);
          if (f < ua.cap) {
            forced_list[f] = slot;
            ua.diverged[f] = 0u;
          } else {
            f = kNone;
          }
        }
        uint32_t* rec = state + (size_t)slot * kPStateWords;
        rec[0] = (uint32_t)sp;
        rec[1] = visits;
        rec[2] = f != kNone ? forcer : kNone;
        rec[3] = f;
      }
      *s_slot = slot;
    }
    __syncthreads();
    const uint32_t slot = *s_slot;
    if (slot >= handoff_cap) return false;
    uint32_t* rec = state + (size_t)slot * kPStateWords;
    for (int k = (int)threadIdx.x; k < sp; k += kPT * kS) rec[4 + k] = s_stack[k];
    if (forcer != kNone && rec[3] != kNone) ua.head[rec[3] * (uint32_t)kPT + (uint32_t)ray] = kNone;
    return true;
  };
  if (may_hand_off) {  // a packet holding a ray that passes every box test visits every node: at once
    if (threadIdx.x == 0) *s_slot = kNone;
    __syncthreads();
    if (in_image && part == 0 && crosses_every_box(invdir)) atomicMin(s_slot, (uint32_t)ray);
    __syncthreads();
    const uint32_t forcer = *s_slot;
    if (forcer != kNone) {
      may_hand_off = false;
      if (hand_off(forcer)) return true;
    }
  }
  __syncthreads();
  const float4 dir0 = *s_dir0;
  uint32_t tested = 0;  // block-uniform: faces of the leaves visited, while may_hand_off
  const uint32_t max_visits = 2 * node_count + 2;
  while (sp > 0 && ++visits <= max_visits) {
    const uint32_t nid = s_stack[--sp];
    if (nid >= node_count) break;  // block-uniform; never taken for a tree built by this library
    const NodeRegs nd = load_node(nodes, nid);  // block-uniform address
    if (rk::node_is_leaf(nd.w0)) {
      const uint32_t tri_id = nd.w1;
      const uint32_t cnt = tri_id < face_count ? min(rk::leaf_count(nd.w0), face_count - tri_id) : 0u;
      if (may_hand_off) {
        if (cnt > handoff_faces - tested) {
          may_hand_off = false;
          ++sp;  // the leaf goes back on top (s_stack still holds it), its pop is not counted
          --visits;
          if (hand_off(kNone)) {
            if (in_image && part == 0) {
              faces_id[l] = fid;
              coords[l] = coord;
              depths[l] = depth;
            }
            return true;
          }
          --sp;
          ++visits;
        } else {
          tested += cnt;
        }
      }
      if (kS == 1) {
        if (in_image) {
          if (cnt <= kGroup && mesh.tris) uniform_leaf(mesh, tri_id, tri_id + cnt, orig, dir, depth, fid, coord);
          else lane_leaf(mesh, tri_id, cnt, orig, dir, cr, depth, fid, coord);
        }
      } else {
        // part p: an equal run of the leaf's faces, or of its groups of faces
        const uint32_t end = tri_id + cnt, unit = cnt <= kPlainLeaf ? 1u : kGroup, g_first = tri_id / unit;
        const uint32_t ng = cnt ? (end - 1u) / unit + 1u - g_first : 0u, q = (ng + kS - 1) / kS;
        const uint32_t ga = min((uint32_t)part * q, ng), gb = min(ga + q, ng);
        float pt = depth;
        float2 puv = make_float2(0.0f, 0.0f);
        uint32_t pk = 0xffffffffu;  // none
        if (in_image && ga < gb) {
          const uint32_t a = max(tri_id, (g_first + ga) * unit);
          const uint32_t m = gb == ng ? end - a : (g_first + gb) * unit - a;
          if (unit == 1u) plain_leaf<kPlainBatch>(mesh, a, a + m, orig, dir, pt, pk, puv);
          else lane_leaf(mesh, a, m, orig, dir, cr, pt, pk, puv);
        }
        s_pt[threadIdx.x] = pt;
        s_pu[threadIdx.x] = puv.x;
        s_pv[threadIdx.x] = puv.y;
        s_pk[threadIdx.x] = pk;
        __syncthreads();
        if (in_image) {
#pragma unroll
          for (int p = 0; p < kS; ++p) {
            const int o = p * kPT + ray;
            const uint32_t k = s_pk[o];
            if (k != 0xffffffffu && s_pt[o] < depth) {
              depth = s_pt[o];
              fid = k;
              coord = make_float2(s_pu[o], s_pv[o]);
            }
          }
        }
        __syncthreads();
      }
    } else {
      int hit = 0;
      if (in_image) {
        float t;
        if (box_ray(nd.bmin, nd.bmax, orig, invdir, t) && t < depth) hit = 1;
      }
      const int any = __syncthreads_or(hit);
      if (any) {
        uint32_t nearc, farc;
        children_order(nd.w0, nd.w1, dir0, nearc, farc);
        if (sp + 2 > kPStack) break;  // block-uniform; cannot occur for trees of depth <= 126
        if (threadIdx.x == 0) { s_stack[sp] = farc; s_stack[sp + 1] = nearc; }
        sp += 2;
      }
      __syncthreads();
    }
  }
  if (in_image && part == 0) {
    faces_id[l] = fid;
    coords[l] = coord;
    depths[l] = depth;
  }
  return false;
}

// The packet traversal's first pass: one 192-thread block per packet.
__global__ __launch_bounds__(kPT) void k_trace_packet(const rk::Node* __restrict__ nodes,
                                                      RefMesh mesh,
                                                      const float4* __restrict__ origins,
                                                      const float4* __restrict__ dirs, int width, int height,
                                                      uint32_t node_count, uint32_t face_count,
                                                      uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                      float* __restrict__ depths, uint32_t* __restrict__ handoff,
                                                      uint32_t handoff_cap, uint32_t handoff_faces,
                                                      uint32_t* __restrict__ forced_list, UnitArgs ua) {
  __shared__ uint32_t s_stack[kPStack];
  __shared__ float4 s_dir0;
  __shared__ uint32_t s_slot;
  trace_packet_job<1>(nodes, mesh, origins, dirs, width, height, node_count, face_count, faces_id, coords,
                      depths, (int)blockIdx.x, (int)blockIdx.y, handoff, handoff_cap, handoff_faces,
                      handoff + kHandoffHead + handoff_cap, forced_list, ua, nullptr, s_stack, &s_dir0,
                      &s_slot, nullptr, nullptr, nullptr, nullptr);
}

// The second pass: the packets handed off, each resumed from its record,
// kPacketSplit threads per ray.
#ifndef RK_REF_PACKET_SPLIT
#define RK_REF_PACKET_SPLIT 5
#endif
constexpr int kPacketSplit = RK_REF_PACKET_SPLIT;

__global__ __launch_bounds__(kPT * kPacketSplit) void k_trace_packet_split(
    const rk::Node* __restrict__ nodes, RefMesh mesh,
    const float4* __restrict__ origins, const float4* __restrict__ dirs, int width, int height, int packets_x,
    uint32_t node_count, uint32_t face_count, const uint32_t* __restrict__ handoff, uint32_t handoff_cap,
    uint32_t* __restrict__ faces_id, float2* __restrict__ coords, float* __restrict__ depths) {
  __shared__ uint32_t s_stack[kPStack];
  __shared__ float4 s_dir0;
  __shared__ uint32_t s_slot;
  __shared__ float s_pt[kPT * kPacketSplit], s_pu[kPT * kPacketSplit], s_pv[kPT * kPacketSplit];
  __shared__ uint32_t s_pk[kPT * kPacketSplit];
  const uint32_t count = min(handoff[0], handoff_cap);
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const uint32_t pk = handoff[kHandoffHead + i];
    const uint32_t* rec = handoff + kHandoffHead + handoff_cap + (size_t)i * kPStateWords;
    if (rec[3] == kDone) continue;  // traced by the forced walk
    trace_packet_job<kPacketSplit>(nodes, mesh, origins, dirs, width, height, node_count, face_count,
                                   faces_id, coords, depths, (int)(pk % (uint32_t)packets_x),
                                   (int)(pk / (uint32_t)packets_x), nullptr, 0u, 0u, nullptr, nullptr, UnitArgs{}, rec,
                                   s_stack, &s_dir0, &s_slot, s_pt, s_pu, s_pv, s_pk);
    __syncthreads();  // the next packet rewrites the stack and s_dir0
  }
}

// The forced packets' results: into the outputs (and the packet's record
// marked kDone) when no walk diverged, the pops keep to the visit limit and
// the forcing ray's final depth is above 0 (then it was above 0 all along);
// otherwise k_trace_packet_split walks the packet from its record.
constexpr uint32_t kForcedCap = 1024;  // forced packets per call
constexpr uint32_t kHitsPerSlot = 2;   // hit entries per forced packet's ray on average
constexpr uint32_t kHitsPerRay = 32;   // and per crossing ray

__global__ __launch_bounds__(kPT) void k_packet_commit(uint32_t node_count, const float4* __restrict__ dirs,
                                                       uint32_t* __restrict__ handoff, UnitArgs ua, PacketArgs pa,
                                                       uint32_t* __restrict__ faces_id, float2* __restrict__ coords,
                                                       float* __restrict__ depths) {
  __shared__ uint32_t s_ok;
  const uint32_t nf = min(handoff[2], ua.cap);
  const uint64_t max_visits = 2 * node_count + 2;
  for (uint32_t f = blockIdx.x; f < nf; f += gridDim.x) {
    const uint32_t slot = pa.forced[f];
    uint32_t* rec = handoff + kHandoffHead + pa.handoff_cap + (size_t)slot * kPStateWords;
    const uint32_t pk = handoff[kHandoffHead + slot];
    const int x0 = (int)(pk % (uint32_t)pa.packets_x) * kPW, y0 = (int)(pk / (uint32_t)pa.packets_x) * kPH;
    const uint32_t q = threadIdx.x;
    const int x = x0 + (int)q % kPW, y = y0 + (int)q / kPW;
    const bool in_image = x < pa.width && y < pa.height;
    const uint32_t l = in_image ? (uint32_t)y * (uint32_t)pa.width + (uint32_t)x : 0u;
    UnitHit h;
    const bool hit = in_image && unit_best(ua, f * (uint32_t)kPT + q, h);
    if (q == rec[2]) {
      const uint32_t o = octant_of(dirs[(uint32_t)y0 * (uint32_t)pa.width + (uint32_t)x0]);
      bool ok = ua.diverged[f] == 0u && (hit ? h.t : depths[l]) > 0.0f;
      for (uint32_t w = 0; w < kPGroups; ++w) ok = ok && ua.pops[f * kPGroups + w] + ua.cut->tops[o] <= max_visits;
      s_ok = ok ? 1u : 0u;
    }
    __syncthreads();  // also: every thread has read the record before it is marked
    if (s_ok != 0u) {
      if (hit) {
        faces_id[l] = h.face;
        coords[l] = make_float2(h.u, h.v);
        depths[l] = h.t;
      }
      if (q == 0) rec[3] = kDone;
    }
    __syncthreads();  // s_ok is read before the next packet's
  }
}

}  // namespace

#ifndef RK_REF_PACKET_HANDOFF_FACES
#define RK_REF_PACKET_HANDOFF_FACES 4096
#endif
constexpr uint32_t kPacketGrid = 1024;  // blocks of the packet traversal's second pass

static std::atomic<uint32_t> g_ray_faces{RK_HANDOFF_AUTO};
static std::atomic<uint32_t> g_packet_faces{RK_HANDOFF_AUTO};
// RK_HANDOFF_AUTO: below 2^19 rays the first pass holds fewer waves than the
// GPU runs at once (about 5,000), and rays handed off early to a wave of their
// own finish sooner: on a 179k-face heightfield a 512x512 per-ray frame takes
// 0.69 ms past 256 faces against 1.23 past 4096, a packet frame 0.87 past 512
// against 1.17. On the 1M-face heightfield at 1920x1080 it is 3.33 against 1.83
// and 3.78 against 3.27. Which is better below 2^19 rays depends on the view, which
// a rule by sizes does not see (per-ray, 256 against 4096): the 20k-face icosphere at
// 512x512 1.02 and 0.50 ms, from twice as far 0.57 and 0.71; 30,000 scattered faces at
// 704x545 5.31 and 2.72, from twice as far 1.63 and 3.16. Of 570 random per-ray
// frames early left one slower than testing every face, late from 12 rays per face on
// many (the last: 2.06).
constexpr uint32_t kAutoRaysBelow = 1u << 19;
constexpr uint32_t kAutoSmallRayFaces = 256, kAutoSmallPacketFaces = 512;
static uint32_t limit_of(uint32_t set, uint32_t n_rays, uint32_t small_limit, uint32_t large_limit) {
  if (set != RK_HANDOFF_AUTO) return set;
  return n_rays < kAutoRaysBelow ? small_limit : large_limit;
}
static std::atomic<uint32_t> g_list_cap{kHandoffCap};
constexpr uint32_t kNoHandoff = 0xffffffffu;

// A memory pool per device for the hand-off buffers, which keeps what calls
// free (the default pool returns it at every synchronisation, and the next
// call would allocate again: 0.3-1 ms per call on the 1920x1080 frame).
static std::mutex g_pool_mutex;
static hipMemPool_t g_pools[64];
static bool g_pool_tried[64];

static hipMemPool_t handoff_pool() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  if (!g_pool_tried[dev]) {
    g_pool_tried[dev] = true;
    hipMemPoolProps props{};
    props.allocType = hipMemAllocationTypePinned;
    props.handleTypes = hipMemHandleTypeNone;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    hipMemPool_t pool = nullptr;
    if (hipMemPoolCreate(&pool, &props) == hipSuccess) {
      uint64_t keep = UINT64_MAX;
      if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess) {
        g_pools[dev] = pool;
      } else {
        (void)hipMemPoolDestroy(pool);
      }
    }
    (void)hipGetLastError();
  }
  return g_pools[dev];
}

// The hand-off buffer of one call (words 32-bit words), its counters and its
// groups' pops (at word pops_off) cleared, the tree's cut made (at cut_off):
// a stream-ordered allocation, so that calls on other streams have their own.
// Without it (nullptr) every ray or packet stays in the first pass, with the
// same results.
static uint32_t* handoff_alloc(hipStream_t st, size_t words, size_t pops_off, uint32_t groups, size_t cut_off,
                               const rk_bvnode* nodes, uint32_t node_count, uint32_t faces) {
  uint32_t* ho = nullptr;
  if (faces == kNoHandoff || words <= kHandoffHead) return nullptr;
  hipMemPool_t pool = handoff_pool();
  const size_t bytes = words * sizeof(uint32_t);
  const hipError_t e = pool ? hipMallocFromPoolAsync(reinterpret_cast<void**>(&ho), bytes, pool, st)
                            : hipMallocAsync(reinterpret_cast<void**>(&ho), bytes, st);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  hipLaunchKernelGGL(k_units_cut, dim3(8 + (std::max(groups, kHandoffHead) + 255) / 256), dim3(256), 0, st,
                     reinterpret_cast<const rk::Node*>(nodes), node_count, reinterpret_cast<UnitCut*>(ho + cut_off), ho,
                     reinterpret_cast<unsigned long long*>(ho + pops_off), groups);
  return ho;
}

#ifndef RK_REF_TRI_RECORDS
#define RK_REF_TRI_RECORDS 1
#endif

// The call's triangle records and group bounds (k_tri_records), one block from
// the same pool; without it the kernels read the faces and vertices.
static RefMesh ref_mesh_alloc(hipStream_t st, const uint4* faces, const float4* verts, uint32_t face_count) {
  RefMesh m{faces, verts, nullptr, nullptr, nullptr};
  if (!RK_REF_TRI_RECORDS) return m;
  char* block = nullptr;
  hipMemPool_t pool = handoff_pool();
  const size_t rec_bytes = rk_align_up((size_t)face_count * kRecFloats * sizeof(float));
  const size_t n_groups = ((size_t)face_count + kGroup - 1) / kGroup;
  const size_t bytes = rec_bytes + (n_groups + ((size_t)face_count + 63) / 64) * sizeof(rk::FaceBound);
  const hipError_t e = pool ? hipMallocFromPoolAsync(reinterpret_cast<void**>(&block), bytes, pool, st)
                            : hipMallocAsync(reinterpret_cast<void**>(&block), bytes, st);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return m;
  }
  float* tris = reinterpret_cast<float*>(block);
  rk::FaceBound* bounds = reinterpret_cast<rk::FaceBound*>(block + rec_bytes);
  hipLaunchKernelGGL(k_tri_records, dim3((face_count + 255) / 256), dim3(256), 0, st, faces, verts, face_count, tris,
                     bounds, bounds + n_groups);
  m.tris = tris;
  m.bounds = bounds;
  m.supers = bounds + n_groups;
  return m;
}

extern "C" rk_status rk_raytrace_mesh_tree(rk_stream stream, const rk_bvnode* nodes, uint32_t node_count,
                                           const rk_uint4* faces, uint32_t face_count, const rk_float4* vertices,
                                           const rk_float4* origins,
                                           const rk_float4* directions, int width, int height, uint32_t* faces_id,
                                           rk_float2* coords, float* depths, int coherency) {
  if (width <= 0 || height <= 0) return RK_ERROR_INVALID_VALUE;
  if (!nodes || node_count == 0 || !faces || face_count == 0 || !vertices || !origins || !directions || !faces_id || !coords || !depths)
    return RK_ERROR_INVALID_VALUE;
  hipStream_t st = rk_hip_stream(stream);
  const uint32_t n = (uint32_t)width * (uint32_t)height;
  if (coherency) {
    // A packet whose leaves pass g_packet_faces faces is traced on by the second
    // pass, kPacketSplit threads per ray, from where it was left. One holding a ray
    // that passes every box test (the packet then visits every leaf, and all its
    // rays test every face) goes at once to walks split by subtree (k_unit_walk,
    // k_packet_commit), and to the second pass when these do not take it or diverge.
    const uint32_t gx = (uint32_t)(width + kPW - 1) / kPW, gy = (uint32_t)(height + kPH - 1) / kPH;
    const uint32_t faces_limit = limit_of(g_packet_faces.load(std::memory_order_relaxed), n, kAutoSmallPacketFaces,
                                          RK_REF_PACKET_HANDOFF_FACES);
    const uint32_t cap = std::min<uint32_t>(gx * gy, g_list_cap.load(std::memory_order_relaxed));
    const uint32_t fcap = std::min<uint32_t>(cap, kForcedCap);
    // [head | list | records | pops (2 words each) | forced list | diverged | slots' heads | cut | hit entries]
    const size_t pops_off = (kHandoffHead + (size_t)cap * (1u + kPStateWords) + 1) & ~size_t(1);
    const size_t flist_off = pops_off + 2ull * kPGroups * fcap;
    const size_t cut_off = flist_off + (2ull + kPT) * fcap;
    const size_t hits_off = cut_off + sizeof(UnitCut) / 4;
    const uint32_t hit_cap = kHitsPerSlot * kPT * fcap;
    uint32_t* ho = handoff_alloc(st, hits_off + hit_cap * (sizeof(UnitHit) / 4), pops_off, kPGroups * fcap, cut_off,
                                 nodes, node_count, faces_limit);
    UnitArgs ua{};
    PacketArgs pa{width, height, (int)gx, cap, ho ? ho + flist_off : nullptr};
    if (ho) {
      ua.pops = reinterpret_cast<unsigned long long*>(ho + pops_off);
      ua.diverged = ho + flist_off + fcap;
      ua.head = ho + flist_off + 2ull * fcap;
      ua.cut = reinterpret_cast<UnitCut*>(ho + cut_off);
      ua.hits = reinterpret_cast<UnitHit*>(ho + hits_off);
      ua.cap = fcap;
      ua.hit_cap = hit_cap;
    }
    const rk::Node* nd = reinterpret_cast<const rk::Node*>(nodes);
    const float4* org = reinterpret_cast<const float4*>(origins);
    const float4* drs = reinterpret_cast<const float4*>(directions);
    float2* uv = reinterpret_cast<float2*>(coords);
    const RefMesh mesh = ref_mesh_alloc(st, reinterpret_cast<const uint4*>(faces),
                                        reinterpret_cast<const float4*>(vertices), face_count);
    hipLaunchKernelGGL(k_trace_packet, dim3(gx, gy), dim3(kPT), 0, st, nd, mesh, org, drs, width, height, node_count,
                       face_count, faces_id, uv, depths, ho, ho ? cap : 0u, faces_limit, ho ? ho + flist_off : nullptr,
                       ua);
    if (ho) {
      hipLaunchKernelGGL(k_unit_walk<true>, dim3(kUnitGrid), dim3(64), 0, st, nd, mesh, org, drs, depths, node_count,
                         face_count, ho, ua, pa);
      hipLaunchKernelGGL(k_packet_commit, dim3(fcap), dim3(kPT), 0, st, node_count, drs, ho, ua, pa, faces_id, uv,
                         depths);
      hipLaunchKernelGGL(k_trace_packet_split, dim3(std::min<uint32_t>(cap, kPacketGrid)), dim3(kPT * kPacketSplit),
                         0, st, nd, mesh, org, drs, width, height, (int)gx, node_count, face_count, ho, cap, faces_id,
                         uv, depths);
      if (hipFreeAsync(ho, st) != hipSuccess) return RK_ERROR_DEVICE;
    }
    if (mesh.tris && hipFreeAsync(const_cast<float*>(mesh.tris), st) != hipSuccess) return RK_ERROR_DEVICE;
  } else {
    // A ray whose leaves pass g_ray_faces faces is traced again by the second
    // pass, one wave per ray. A ray that passes every box test goes at once to walks
    // split by subtree (k_unit_walk, k_units_merge), and to the second pass when these
    // do not take it (then at its first leaf) or diverge.
    const uint32_t faces_limit = limit_of(g_ray_faces.load(std::memory_order_relaxed), n, kAutoSmallRayFaces,
                                          RK_REF_HANDOFF_FACES);
    const uint32_t cap = std::min<uint32_t>(n, g_list_cap.load(std::memory_order_relaxed));
    const uint32_t ucap = std::min<uint32_t>(cap, kCrossCap);
    // [head | list | pops (2 words each) | crossing rays: list, buckets (8), redo, diverged, heads | cut | hit entries]
    const uint32_t groups = ucap / 64 + 8;
    const size_t pops_off = (kHandoffHead + cap + 1ull) & ~size_t(1);
    const size_t list_off = pops_off + 2ull * groups;
    const size_t cut_off = list_off + 12ull * ucap;
    const size_t hits_off = cut_off + sizeof(UnitCut) / 4;
    const uint32_t hit_cap = kHitsPerRay * ucap;
    uint32_t* ho = handoff_alloc(st, hits_off + hit_cap * (sizeof(UnitHit) / 4), pops_off, groups, cut_off, nodes,
                                 node_count, faces_limit);
    UnitArgs ua{};
    if (ho) {
      uint32_t* p = ho + list_off;
      ua.pops = reinterpret_cast<unsigned long long*>(ho + pops_off);
      ua.list = p;
      ua.bucket = p + ucap;
      ua.redo = p + 9ull * ucap;
      ua.diverged = p + 10ull * ucap;
      ua.head = p + 11ull * ucap;
      ua.cut = reinterpret_cast<UnitCut*>(ho + cut_off);
      ua.hits = reinterpret_cast<UnitHit*>(ho + hits_off);
      ua.cap = ucap;
      ua.hit_cap = hit_cap;
    }
    const rk::Node* nd = reinterpret_cast<const rk::Node*>(nodes);
    const float4* org = reinterpret_cast<const float4*>(origins);
    const float4* drs = reinterpret_cast<const float4*>(directions);
    float2* uv = reinterpret_cast<float2*>(coords);
    const RefMesh mesh = ref_mesh_alloc(st, reinterpret_cast<const uint4*>(faces),
                                        reinterpret_cast<const float4*>(vertices), face_count);
    const uint32_t w = (uint32_t)width, tiles_x = tiled_rays(w, (uint32_t)height) ? (w + kTileW - 1) / kTileW : 0u;
    const uint32_t blocks = tiles_x ? tiles_x * (((uint32_t)height + kTileH - 1) / kTileH) : (n + 63) / 64;
    hipLaunchKernelGGL(k_trace_ray<RK_REF_COOP_MAX>, dim3(blocks), dim3(64), 0, st, nd, mesh, org, drs, n, w,
                       (uint32_t)height, tiles_x, node_count, face_count, faces_id, uv, depths, ho, ho ? cap : 0u,
                       faces_limit, ua);
    if (ho) {
      hipLaunchKernelGGL(k_unit_walk<false>, dim3(kUnitGrid), dim3(64), 0, st, nd, mesh, org, drs, depths, node_count,
                         face_count, ho, ua, PacketArgs{});
      hipLaunchKernelGGL(k_units_merge, dim3((ucap + 63) / 64), dim3(64), 0, st, node_count, ho, ua, faces_id, uv,
                         depths);
      hipLaunchKernelGGL(k_trace_ray_wave, dim3(std::min<uint32_t>(cap, kRayWaveGrid)), dim3(64), 0, st, nd, mesh,
                         org, drs, node_count, face_count, ho, cap, ua.redo, ucap, faces_id, uv, depths);
      if (hipFreeAsync(ho, st) != hipSuccess) return RK_ERROR_DEVICE;
    }
    if (mesh.tris && hipFreeAsync(const_cast<float*>(mesh.tris), st) != hipSuccess) return RK_ERROR_DEVICE;
  }
  RK_CHECK_LAUNCH();
  return RK_SUCCESS;
}

extern "C" rk_status rk_raytrace_set_handoff(uint32_t ray_faces, uint32_t packet_faces, uint32_t list_cap) {
  if (list_cap == 0 || list_cap > kHandoffCap) return RK_ERROR_INVALID_VALUE;
  g_ray_faces.store(ray_faces, std::memory_order_relaxed);
  g_packet_faces.store(packet_faces, std::memory_order_relaxed);
  g_list_cap.store(list_cap, std::memory_order_relaxed);
  return RK_SUCCESS;
}

extern "C" rk_status rk_raytrace_get_handoff(uint32_t* ray_faces, uint32_t* packet_faces, uint32_t* list_cap) {
  if (!ray_faces || !packet_faces || !list_cap) return RK_ERROR_INVALID_VALUE;
  *ray_faces = g_ray_faces.load(std::memory_order_relaxed);
  *packet_faces = g_packet_faces.load(std::memory_order_relaxed);
  *list_cap = g_list_cap.load(std::memory_order_relaxed);
  return RK_SUCCESS;
}
