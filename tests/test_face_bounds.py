"""The bounds that let the reference traversals skip groups of faces: on the CPU
against the triangle test itself, and on the GPU at the edges of a group (16
faces) and of a wave's faces (64)."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
F32MAX = np.finfo(np.float32).max

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "rk_face_bounds.h"
static uint64_t s = 88172645463325252ull;
static double u01() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return (double)(s >> 11) * (1.0 / 9007199254740992.0); }
static double sym() { return 2.0 * u01() - 1.0; }
struct V { float x, y, z; };
static V sub(V a, V b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
static V cross(V a, V b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
static float dot(V a, V b) { return a.x * b.x + a.y * b.y + a.z * b.z + 0.0f; }
static bool tri_ray(V o, V d, V v0, V e1, V e2, float& t) {  // the reference's, w = 0
  V p = cross(d, e2);
  float det = dot(e1, p);
  if (det > -0.000001f && det < 0.000001f) return false;
  float inv = 1.0f / det;
  V tv = sub(o, v0);
  float u = dot(tv, p) * inv;
  if (u < 0.0f || u > 1.0f) return false;
  V q = cross(tv, e1);
  float v = dot(d, q) * inv;
  if (v < 0.0f || u + v > 1.0f) return false;
  t = dot(e2, q) * inv;
  return t >= 0.0f;
}
int main(int argc, char** argv) {
  const long trials = atol(argv[1]);
  long accepted = 0, outside = 0, missed = 0, lost = 0;
  for (long n = 0; n < trials; ++n) {
    const double scale = pow(10.0, -3.0 + 5.0 * u01()), far = scale * pow(10.0, 4.0 * u01() - 1.0);
    const int faces = 1 + (int)(u01() * 16);
    V a[16], b[16], c[16];
    float lo[3], hi[3], e2m = 0;
    for (int k = 0; k < 3; ++k) { lo[k] = INFINITY; hi[k] = -INFINITY; }
    const double off[3] = {far * sym(), far * sym(), far * sym()};
    for (int f = 0; f < faces; ++f) {
      V* p[3] = {&a[f], &b[f], &c[f]};
      const double thin = u01() < 0.4 ? pow(10.0, -6.0 * u01()) : 1.0;  // slivers
      double q[3][3];
      for (int k = 0; k < 3; ++k) { q[0][k] = off[k] + 4 * scale * sym(); q[1][k] = q[0][k] + scale * sym(); }
      for (int k = 0; k < 3; ++k) q[2][k] = q[0][k] + (q[1][k] - q[0][k]) * u01() + thin * scale * sym();
      for (int k = 0; k < 3; ++k) *p[k] = {(float)q[k][0], (float)q[k][1], (float)q[k][2]};
      for (int k = 0; k < 3; ++k) {
        const float w[3] = {p[k]->x, p[k]->y, p[k]->z};
        for (int j = 0; j < 3; ++j) { lo[j] = fminf(lo[j], w[j]); hi[j] = fmaxf(hi[j], w[j]); }
      }
      V e1 = sub(b[f], a[f]), e2 = sub(c[f], a[f]);
      e2m = fmaxf(e2m, fmaxf(dot(e1, e1), dot(e2, e2)));
    }
    const rk::FaceBound bound = rk::face_bound(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], 1.00001f * e2m);
    for (int r = 0; r < 8; ++r) {
      // a ray through a point of a face's plane at or just past an edge, at a
      // slope down to the one where |det| meets the threshold
      const int f = (int)(u01() * faces);
      const double wu = u01() * 1.2 - 0.1, wv = (1.0 - wu) * (u01() * 1.2 - 0.1);
      V e1 = sub(b[f], a[f]), e2 = sub(c[f], a[f]);
      const double P[3] = {a[f].x + wu * e1.x + wv * e2.x, a[f].y + wu * e1.y + wv * e2.y, a[f].z + wu * e1.z + wv * e2.z};
      const double slope = u01() < 0.5 ? pow(10.0, -6.0 * u01()) : 1.0, len = pow(10.0, 2.0 * u01() - 1.0);
      const double i = sym(), j = sym();
      double D[3] = {i * e1.x + j * e2.x + slope * scale * sym(), i * e1.y + j * e2.y + slope * scale * sym(),
                     i * e1.z + j * e2.z + slope * scale * sym()};
      const double dn = sqrt(D[0] * D[0] + D[1] * D[1] + D[2] * D[2]), dist = scale * pow(10.0, 3.0 * u01() - 1.0);
      if (!(dn > 0)) continue;
      if (u01() < 0.2) D[(int)(u01() * 3)] = 0.0;
      const V d = {(float)(D[0] / dn * len), (float)(D[1] / dn * len), (float)(D[2] / dn * len)};
      const V o = {(float)(P[0] - D[0] / dn * dist), (float)(P[1] - D[1] / dn * dist), (float)(P[2] - D[2] / dn * dist)};
      const rk::CullRay cr = rk::cull_ray(o.x, o.y, o.z, 0.0f, d.x, d.y, d.z, 0.0f);
      for (int g = 0; g < faces; ++g) {
        float t;
        if (!tri_ray(o, d, a[g], sub(b[g], a[g]), sub(c[g], a[g]), t)) continue;
        ++accepted;
        const float past = nextafterf(t, INFINITY);  // the smallest depth that keeps the hit
        if (rk::bound_missed(bound, o.x, o.y, o.z, d.x, d.y, d.z, cr, past)) ++lost;
        const double h[3] = {o.x + (double)t * d.x, o.y + (double)t * d.y, o.z + (double)t * d.z};
        for (int k = 0; k < 3; ++k) if (h[k] < lo[k] || h[k] > hi[k]) { ++outside; break; }
      }
      const V e = {(float)(o.x + 20 * scale * sym()), (float)(o.y + 20 * scale * sym()), (float)(o.z + 20 * scale * sym())};
      if (rk::bound_missed(bound, e.x, e.y, e.z, d.x, d.y, d.z, cr, 3e38f)) ++missed;
    }
    // never skipped: values that are not finite or too large
    const float bad[4] = {NAN, INFINITY, -INFINITY, 2e9f}, x = bad[n & 3];
    const rk::CullRay cr = rk::cull_ray(0, x, 0, 0, 1, 1, 1, 0), cd = rk::cull_ray(0, 0, 0, 0, 1, x, 1, 0);
    const rk::CullRay ok = rk::cull_ray(9, 9, 9, 0, 1, 0, 0, 0), tiny = rk::cull_ray(9, 9, 9, 0, 1e-23f, 0, 0, 0);
    const rk::FaceBound wide = rk::face_bound(lo[0], lo[1], lo[2], x, hi[1], hi[2], e2m);
    const rk::FaceBound edge = rk::face_bound(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], (n & 3) == 3 ? INFINITY : x * x);
    if (rk::bound_missed(bound, 0, x, 0, 1, 1, 1, cr, 1) || rk::bound_missed(bound, 0, 0, 0, 1, x, 1, cd, 1) ||
        rk::bound_missed(bound, 9, 9, 9, 1e-23f, 0, 0, tiny, 3e38f) ||
        ((n & 3) != 0 && rk::bound_missed(wide, 9, 9, 9, 1, 0, 0, ok, 1)) || rk::bound_missed(edge, 9, 9, 9, 1, 0, 0, ok, 1))
      ++lost;
  }
  printf("%ld %ld %ld %ld\n", accepted, outside, missed, lost);
  return 0;
}
"""


def test_bounds_keep_every_accepted_face(tmp_path):
    """No face that the reference's float test accepts lies in a group the bound
    skips, over slivers, grazing rays at the |det| threshold, rays with zero
    components and depths just past the hit."""
    src, exe = tmp_path / "bounds.cpp", tmp_path / "bounds"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", f"-I{ROOT / 'cudart_amd' / 'csrc'}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe), "150000"], check=True, capture_output=True, text=True, timeout=100).stdout
    accepted, outside, missed, lost = map(int, out.split())
    assert lost == 0
    assert accepted > 100_000 and outside > 100 and missed > 100_000  # hits past the box, and bounds that do skip


@pytest.mark.gpu
@pytest.mark.parametrize("packet", [False, True])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 48, 63, 64, 65, 257, 1025])
def test_trace_at_group_edges(rk, ora, n, packet):
    """Meshes around a group's and a wave's number of faces, as one leaf and as a
    tree, with rays that pass every box test among the others: bit-exact."""
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(n, seed=n, mu=float(np.log(0.3)))
    hb = rk.hitbox(V)
    w, h = 37, 26
    O, D = rk.random_rays(w * h, seed=n + 1)
    D[::7, 1] = 0.0
    for depth in (0, 8):
        ref = ora.build_lbvh_ref(F, V, hb, depth, True)
        Ft, Vt = torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda()
        tree = dev.build_lbvh(Ft, Vt, hb, depth, True)
        out = dev.trace_ref(tree, Vt, torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda(), w, h, packet)
        if packet:
            of, ouv, od, _ = ora.trace_ref_packet(ref.nodes, ref.faces, V, O, D, w, h)
        else:
            of, ouv, od, _ = ora.trace_ref_ray(ref.nodes, ref.faces, V, O, D)
        got = [t.cpu().numpy() for t in out]
        np.testing.assert_array_equal(got[0].view(np.uint32), of)
        np.testing.assert_array_equal(got[1], ouv)
        np.testing.assert_array_equal(got[2], od)
