// Conservative bounds of groups of faces for the reference triangle test: a
// group whose bound a ray misses holds no face that tri_ray (the reference's
// float arithmetic, CUDA_raytraceMeshTree.cu:57-89, |det| >= 1e-6) accepts
// with t < depth, so skipping it changes no result. Plain C++ so that the
// host tests compile the same code as the kernels.
//
// Why it holds. Let u = 2^-24, tvec = orig - v0, and let det, un, vn, tn be
// the computed determinant and numerators. Standard error bounds of the
// cross and dot products give |det - D| <= 7u|e1||e2||d|, and errors of un,
// vn, tn of at most 8u|tvec||d||e2|, 8u|tvec||d||e1| and 8u|tvec||e1||e2|.
// With the true numerators divided by the computed det, Cramer's identity
// puts the point orig + c d (c = tn / det) at v0 + a e1 + b e2 plus at most
// |1 - D/det||tvec|, and the acceptance tests keep (a, b) inside the triangle
// up to the errors over |det|. With |det| >= 1e-6 and E the longest edge from
// v0, the point lies within 5uE + 55e6 u E^2 |d||tvec| = 5uE + 3.28 E^2 |d||tvec|
// of the triangle, and c in [-0.48 E^2 |tvec|, depth (1 + 4u) + 0.48 E^2 |tvec|].
// So an accepted ray meets the group's box grown by that distance; the second
// term's coefficient is taken as 4.04, which covers the slack of c too, and
// 2e-6 of the distance covers the rounding of the test below. Magnitudes up
// to 1e9 keep every product finite; a group or a ray beyond that (or NaN, or a
// direction shorter than 1e-15) is never skipped.
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define RK_FB __host__ __device__ __forceinline__
#else
#define RK_FB inline
#endif

namespace rk {

constexpr uint32_t kFaceGroup = 16;  // consecutive faces per bound
constexpr float kFaceBoundMax = 1e9f;

struct FaceBound {
  float cx, cy, cz;  // centre of the group's box
  float k;           // 4.04 E^2
  float hx, hy, hz;  // half extents, rounded up
  float r1;          // hx + hy + hz
};
static_assert(sizeof(FaceBound) == 32, "bound is 32 B");

// The bound of a group from its box (of the faces' vertices) and the largest
// squared edge length e2max from v0. Not finite or too large: a bound that no
// ray misses.
RK_FB FaceBound face_bound(float lox, float loy, float loz, float hix, float hiy, float hiz, float e2max) {
  FaceBound b;
  const float m = fmaxf(fmaxf(fmaxf(fabsf(lox), fabsf(loy)), fabsf(loz)),
                        fmaxf(fmaxf(fabsf(hix), fabsf(hiy)), fabsf(hiz)));
  if (!(m <= kFaceBoundMax) || !(e2max <= 4.0f * kFaceBoundMax * kFaceBoundMax)) {
    b.cx = b.cy = b.cz = 0.0f;
    b.k = b.hx = b.hy = b.hz = b.r1 = INFINITY;
    return b;
  }
  const float pad = 1e-6f * sqrtf(e2max) + 1e-30f;
  b.cx = 0.5f * (lox + hix);
  b.cy = 0.5f * (loy + hiy);
  b.cz = 0.5f * (loz + hiz);
  b.hx = fmaxf(hix - b.cx, b.cx - lox) * 1.000001f + pad;
  b.hy = fmaxf(hiy - b.cy, b.cy - loy) * 1.000001f + pad;
  b.hz = fmaxf(hiz - b.cz, b.cz - loz) * 1.000001f + pad;
  b.k = 4.04f * e2max;
  b.r1 = b.hx + b.hy + b.hz;
  return b;
}

// A ray's terms for bound_missed: an upper bound of |d| (infinite when the
// ray is not finite or too large, so that nothing is skipped) and |d|^2.
struct CullRay {
  float dl, d2;
};
RK_FB CullRay cull_ray(float ox, float oy, float oz, float ow, float dx, float dy, float dz, float dw) {
  CullRay r;
  const float m = fmaxf(fmaxf(fmaxf(fabsf(ox), fabsf(oy)), fmaxf(fabsf(oz), fabsf(ow))),
                        fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fmaxf(fabsf(dz), fabsf(dw))));
  const float s = ((ox + oy) + (oz + ow)) + ((dx + dy) + (dz + dw));  // NaN when any is (fmaxf drops it)
  r.d2 = dx * dx + dy * dy + dz * dz;
  r.dl = (m <= kFaceBoundMax && s == s && r.d2 >= 1e-30f) ? 1.00001f * sqrtf(r.d2) + 1e-30f : INFINITY;
  return r;
}

// Whether the ray's part [0, depth] misses the group's grown box: the line
// against the box on the three axes across d, then the box's span along d.
// Every comparison is false on NaN, which keeps the group.
RK_FB bool bound_missed(const FaceBound& b, float ox, float oy, float oz, float dx, float dy, float dz,
                        const CullRay& r, float depth) {
  const float wx = b.cx - ox, wy = b.cy - oy, wz = b.cz - oz;
  const float x = ((fabsf(wx) + fabsf(wy)) + fabsf(wz)) + b.r1;
  const float g = x * __builtin_fmaf(b.k, r.dl, 2e-6f);
  const float hx = b.hx + g, hy = b.hy + g, hz = b.hz + g;
  const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
  const float px = __builtin_fmaf(wy, dz, -(wz * dy));
  const float py = __builtin_fmaf(wz, dx, -(wx * dz));
  const float pz = __builtin_fmaf(wx, dy, -(wy * dx));
  const float s = __builtin_fmaf(wx, dx, __builtin_fmaf(wy, dy, wz * dz));
  const float m = __builtin_fmaf(hx, ax, __builtin_fmaf(hy, ay, hz * az));
  bool out = fabsf(px) > __builtin_fmaf(hy, az, hz * ay);
  out = out || fabsf(py) > __builtin_fmaf(hz, ax, hx * az);
  out = out || fabsf(pz) > __builtin_fmaf(hx, ay, hy * ax);
  out = out || s + m < 0.0f;
  out = out || s - m > depth * r.d2;
  return out;
}

}  // namespace rk
