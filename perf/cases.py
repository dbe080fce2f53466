"""Performance cases: the work a program gives this library, through the calls it makes.

Seven kinds, each a call sequence of the public API (cudart_amd.device and, where it
has no wrapper, cudart_amd.native):

  build_fast   rk_fast_build: the throughput tree of a mesh
  trace_fast   rk_fast_trace / rk_fast_trace_sorted: closest hits of a frame's primary
               rays, or of incoherent rays
  animate      rk_fast_refit and rk_fast_render_camera: one frame of a deforming mesh
  build_ref    rk_build_lbvh / rk_build_sah (and both, for Hybrid): the reference trees
  trace_ref    depths cleared, then rk_raytrace_mesh_tree: the reference's per-ray and
               packet traversals
  batch        rk_batch_build, depths cleared, rk_batch_trace: many meshes together
  serve        rk_server_*: a burst of requests over deforming scenes

Scenes are the library's own workloads (icosphere, fBm heightfield, random triangle
soup) made here from a seed with torch alone; cameras are at a 30-degree elevation
with a 60-degree field of view unless drawn otherwise.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from cudart_amd import device as dev
from cudart_amd import native as N
from cudart_amd import scenes

FLT_MAX = float(np.finfo(np.float32).max)


def listed():
    return [
        # The smallest mesh in use: the subdivision-5 icosphere a sample program builds. Launches count.
        {"name": "build_fast_icosphere", "kind": "build_fast", "scene": "icosphere", "size": 5, "morton": 30},
        # An ordinary scene: 999,698 terrain faces, rebuilt when the mesh is loaded or changes.
        {"name": "build_fast_terrain_1m", "kind": "build_fast", "scene": "terrain", "size": 708, "morton": 30},
        # The largest scene: 10M faces, whose density needs 63-bit keys.
        {"name": "build_fast_soup_10m", "kind": "build_fast", "scene": "soup", "size": 10_000_000, "morton": 63},
        # The frame everybody renders: full-HD primary rays of a 1M-face terrain, tree resident.
        {"name": "trace_fast_terrain_1080p", "kind": "trace_fast", "scene": "terrain", "size": 708, "width": 1920,
         "height": 1080, "sorted": False, "azimuth": 45.0, "elevation": 30.0},
        # Secondary, shadow or scattered rays: 16M incoherent rays through 10M faces, in origin order.
        {"name": "trace_fast_soup_sorted_16m", "kind": "trace_fast", "scene": "soup", "size": 10_000_000,
         "rays": 1 << 24, "sorted": True},
        # A small animated object: refit to this frame's vertices and the shaded frame in one launch.
        {"name": "animate_icosphere_256", "kind": "animate", "scene": "icosphere", "size": 5, "width": 256,
         "height": 256, "azimuth": 45.0, "elevation": 30.0},
        # The drop-in path of a program written against the reference: its LBVH at its sample's depth ...
        {"name": "build_ref_lbvh_terrain_1m", "kind": "build_ref", "scene": "terrain", "size": 708, "tree": "lbvh",
         "depth": 12},
        # ... its binned SAH build ...
        {"name": "build_ref_sah_terrain_1m", "kind": "build_ref", "scene": "terrain", "size": 708, "tree": "sah",
         "depth": 12},
        # ... its per-ray traversal ...
        {"name": "trace_ref_ray_terrain_1080p", "kind": "trace_ref", "scene": "terrain", "size": 708, "width": 1920,
         "height": 1080, "packet": False, "depth": 12, "azimuth": 45.0, "elevation": 30.0},
        # ... and its packet traversal (the reference's default) of the same full-HD frame.
        {"name": "trace_ref_packet_terrain_1080p", "kind": "trace_ref", "scene": "terrain", "size": 708,
         "width": 1920, "height": 1080, "packet": True, "depth": 12, "azimuth": 45.0, "elevation": 30.0},
        # Many uneven meshes at once: 1024 of 64 to 65,536 faces, 256 to 16,384 rays each.
        {"name": "batch_1024", "kind": "batch", "meshes": 1024, "max_faces": 65536, "max_rays": 16384, "sorted": False},
        # A burst of requests over deforming scenes of uneven size and resolution.
        {"name": "serve_burst_32", "kind": "serve", "scenes": 8, "max_grid": 400, "requests": 32, "max_side": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_scene(rng, most):
    """A scene of about 1000 faces up to about `most`."""
    kind = rng.choice(["terrain", "terrain", "soup", "icosphere"])
    if kind == "icosphere":
        return kind, rng.choice([k for k in (3, 4, 5, 6, 7) if 20 * 4 ** k <= most])
    if kind == "terrain":
        return kind, _log_int(rng, 24, int(math.sqrt(most / 2)) + 1)
    return kind, _log_int(rng, 1000, most)


def _draw_frame(rng, width, height):
    w = _log_int(rng, 64, width)
    return {"width": w, "height": max(36, min(height, int(w * rng.choice([0.5625, 0.75, 1.0])))),
            "azimuth": rng.choice([45.0, rng.uniform(0.0, 360.0)]),
            "elevation": rng.choice([30.0, rng.uniform(15.0, 60.0)])}


def draw(rng):
    kind = rng.choice(["build_fast", "build_fast", "trace_fast", "trace_fast", "animate", "build_ref", "build_ref",
                       "trace_ref", "trace_ref", "batch", "serve"])
    if kind == "build_fast":
        scene, size = _draw_scene(rng, 5_000_000)
        return {"kind": kind, "scene": scene, "size": size, "morton": rng.choice([30, 30, 63])}
    if kind == "trace_fast":
        scene, size = _draw_scene(rng, 4_000_000)
        if scene == "soup":
            return {"kind": kind, "scene": scene, "size": size, "rays": _log_int(rng, 4096, 4_000_000),
                    "sorted": rng.random() < 0.5}
        return {"kind": kind, "scene": scene, "size": size, "sorted": False, **_draw_frame(rng, 1920, 1080)}
    if kind == "animate":
        scene, size = _draw_scene(rng, 1_000_000)
        return {"kind": kind, "scene": scene, "size": size, **_draw_frame(rng, 1920, 1080)}
    if kind == "build_ref":
        scene, size = _draw_scene(rng, 1_000_000)
        return {"kind": kind, "scene": scene, "size": size, "tree": rng.choice(["lbvh", "lbvh", "sah", "hybrid"]),
                "depth": rng.choice([12, 16, 24, 31])}
    if kind == "trace_ref":
        size = rng.choice([3, 4, 5, 6])
        scene = "icosphere"
        if rng.random() < 0.6:
            scene, size = "terrain", _log_int(rng, 48, 708)
        return {"kind": kind, "scene": scene, "size": size, "packet": rng.random() < 0.5,
                "depth": rng.choice([12, 16, 24]), **_draw_frame(rng, 1920, 1080)}
    if kind == "batch":
        return {"kind": kind, "meshes": _log_int(rng, 16, 1024), "max_faces": _log_int(rng, 512, 65536),
                "max_rays": _log_int(rng, 1024, 16384), "sorted": rng.random() < 0.5}
    return {"kind": kind, "scenes": rng.randint(2, 12), "max_grid": _log_int(rng, 64, 400),
            "requests": rng.randint(4, 48), "max_side": _log_int(rng, 96, 512)}


# ---- scenes --------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 0x9E3779B1 + 12345) % (1 << 62))
    return g


def _with_w(xyz):
    return torch.cat([xyz, torch.zeros_like(xyz[:, :1])], dim=1).float().contiguous()


def _icosphere(levels, seed):
    """The unit icosahedron subdivided `levels` times, in an orientation of the seed's."""
    t = (1 + 5 ** 0.5) / 2
    P = np.array([[-1, t, 0], [1, t, 0], [-1, -t, 0], [1, -t, 0], [0, -1, t], [0, 1, t], [0, -1, -t], [0, 1, -t],
                  [t, 0, -1], [t, 0, 1], [-t, 0, -1], [-t, 0, 1]], np.float64)
    T = np.array([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9], [5, 11, 4], [11, 10, 2],
                  [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2], [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5], [2, 4, 11],
                  [6, 2, 10], [8, 6, 7], [9, 8, 1]], np.int64)
    P /= np.linalg.norm(P, axis=1, keepdims=True)
    for _ in range(levels):
        e = np.sort(np.concatenate([T[:, [0, 1]], T[:, [1, 2]], T[:, [2, 0]]]), axis=1)
        u, inv = np.unique(e[:, 0] * len(P) + e[:, 1], return_inverse=True)
        mid = P[u // len(P)] + P[u % len(P)]
        ab, bc, ca = (len(P) + inv.reshape(-1)).reshape(3, -1)
        P = np.concatenate([P, mid / np.linalg.norm(mid, axis=1, keepdims=True)])
        a, b, c = T.T
        T = np.stack([np.stack(f, 1) for f in ((a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca))], 1).reshape(-1, 3)
    q, _ = np.linalg.qr(np.random.RandomState(seed % (1 << 31)).normal(size=(3, 3)))
    F = np.concatenate([T, np.zeros_like(T[:, :1])], axis=1).astype(np.int32)
    return _with_w(torch.from_numpy(P @ q).cuda()), torch.from_numpy(F).cuda()


def _terrain(grid, seed):
    """grid x grid vertices over the unit square, z a six-octave value-noise fBm scaled to [0, 0.2]."""
    g = _gen(seed)
    x = torch.arange(grid, device="cuda", dtype=torch.float64) / (grid - 1)
    z = torch.zeros(grid, grid, device="cuda", dtype=torch.float64)
    for o in range(6):
        k = 4 << o
        lat = torch.rand(k + 2, k + 2, generator=g, device="cuda", dtype=torch.float64)
        i = (x * k).floor().long().clamp(max=k)
        f = x * k - i
        s = f * f * (3 - 2 * f)
        rows = lat[i] * (1 - s)[:, None] + lat[i + 1] * s[:, None]
        z += 0.5 ** o * (rows[:, i] * (1 - s) + rows[:, i + 1] * s)
    z = 0.2 * (z - z.min()) / (z.max() - z.min())
    V = _with_w(torch.stack([x.repeat(grid), x.repeat_interleave(grid), z.reshape(-1)], dim=1))
    c = torch.arange(grid - 1, device="cuda")
    v = (c[:, None] * grid + c).reshape(-1)
    zero = torch.zeros_like(v)
    F = torch.stack([torch.stack([v, v + 1, v + grid + 1, zero], 1),
                     torch.stack([v, v + grid + 1, v + grid, zero], 1)], 1).reshape(-1, 4)
    return V, F.int().contiguous()


def _soup(n, seed, edge=None):
    """n separate triangles, centroids uniform in the unit cube, edges isotropic with lognormal length (median
    0.002 at 10M faces, scaled to the same total area at other counts)."""
    g = _gen(seed)
    edge = 0.002 * math.sqrt(10_000_000 / n) if edge is None else edge
    c = torch.rand(n, 3, generator=g, device="cuda")
    e = []
    for _ in range(2):
        d = torch.randn(n, 3, generator=g, device="cuda")
        e.append(d / d.norm(dim=1, keepdim=True) * torch.exp(math.log(edge) + 0.5 * torch.randn(n, 1, generator=g,
                                                                                                 device="cuda")))
    v0 = c - (e[0] + e[1]) / 3
    V = _with_w(torch.stack([v0, v0 + e[0], v0 + e[1]], dim=1).reshape(-1, 3))
    F = torch.zeros(n, 4, dtype=torch.int32, device="cuda")
    F[:, :3] = torch.arange(3 * n, dtype=torch.int32, device="cuda").reshape(n, 3)
    return V, F


def _scene(case, seed):
    make = {"icosphere": _icosphere, "terrain": _terrain, "soup": _soup}[case["scene"]]
    return make(case["size"], seed)


def _hitbox(V):
    """The mesh's box, as a program has it from its model."""
    return np.stack([V.amin(0).cpu().numpy(), V.amax(0).cpu().numpy()]).astype(np.float32)


def _faces(case):
    s = case["size"]
    return {"icosphere": 20 * 4 ** s, "terrain": 2 * (s - 1) ** 2, "soup": s}[case["scene"]]


def _vertices(case):
    s = case["size"]
    return {"icosphere": 10 * 4 ** s + 2, "terrain": s * s, "soup": 3 * s}[case["scene"]]


# ---- rays ----------------------------------------------------------------------------


def _camera(case):
    """The orbit camera: 1.5 from a terrain's or a soup's centre, 3 from a sphere's."""
    el, az = math.radians(case["elevation"]), math.radians(case["azimuth"])
    mid, dist = {"terrain": ((0.5, 0.5, 0.1), 1.5), "soup": ((0.5, 0.5, 0.5), 2.0),
                 "icosphere": ((0.0, 0.0, 0.0), 3.0)}[case["scene"]]
    mid = np.array(mid)
    eye = mid + dist * np.array([math.cos(el) * math.cos(az), math.cos(el) * math.sin(az), math.sin(el)])
    return N.camera_lookat(eye, mid, 60 * 0.01745329252, case["width"], case["height"], up=[0, 0, 1])


def _primary(cam, width, height):
    """The camera's rays, (dir - x * step_x) - y * step_y in float32."""
    c = torch.from_numpy(cam).cuda()
    x = torch.arange(width, device="cuda", dtype=torch.float32).repeat(height)[:, None]
    y = torch.arange(height, device="cuda", dtype=torch.float32).repeat_interleave(width)[:, None]
    D = (c[1] - x * c[2]) - y * c[3]
    return c[0].expand(width * height, 4).contiguous(), D.contiguous()


def _scattered(n, seed):
    """Origins uniform in the unit cube, directions uniform on the sphere."""
    g = _gen(seed + 77)
    O = torch.rand(n, 3, generator=g, device="cuda")
    D = torch.randn(n, 3, generator=g, device="cuda")
    return _with_w(O), _with_w(D / D.norm(dim=1, keepdim=True))


def _rays_of(case, seed):
    if "rays" in case:
        return _scattered(case["rays"], seed)
    return _primary(_camera(case), case["width"], case["height"])


def _ray_count(case):
    return case["rays"] if "rays" in case else case["width"] * case["height"]


# ---- prepare and run -----------------------------------------------------------------


def _fast_builder(n, morton):
    b = dev.FastBuilder(n, N.RK_MORTON_63 if morton == 63 else N.RK_MORTON_30)
    b.nodes.zero_()  # one of the n records is not written by a build
    return b


def prepare(case, seed):
    return {"build_fast": _prepare_build_fast, "trace_fast": _prepare_trace_fast, "animate": _prepare_animate,
            "build_ref": _prepare_build_ref, "trace_ref": _prepare_trace_ref, "batch": _prepare_batch,
            "serve": _prepare_serve}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_build_fast(case, seed):
    V, F = _scene(case, seed)
    return {"run": _run_build_fast, "V": V, "F": F, "hitbox": _hitbox(V),
            "builder": _fast_builder(F.shape[0], case["morton"])}


def _run_build_fast(s):
    t = s["builder"].build(s["F"], s["V"], s["hitbox"])
    # the records hold face ids beside coordinates: words, not floats
    return {"nodes": t.nodes, "tris": t.tris.view(torch.int32), "indices": t.indices, "boxes": t.boxes}


def _prepare_trace_fast(case, seed):
    V, F = _scene(case, seed)
    tree = _fast_builder(F.shape[0], 63 if F.shape[0] > 2_000_000 else 30).build(F, V, _hitbox(V))
    O, D = _rays_of(case, seed)
    n = O.shape[0]
    ws = dev.workspace(N.lib().rk_fast_trace_sorted_workspace_size(n)) if case["sorted"] else None
    return {"run": _run_trace_fast, "tree": tree, "O": O, "D": D, "out": dev.new_outputs(n), "ws": ws,
            # the reference's absolute threshold for terrains and spheres; 0 for small scattered triangles
            "eps": 0.0 if case["scene"] == "soup" else None}


def _run_trace_fast(s):
    if s["ws"] is not None:
        out = dev.fast_trace_sorted(s["tree"], s["O"], s["D"], out=s["out"], det_epsilon=s["eps"], ws=s["ws"],
                                    reset_depth=True)
    else:
        out = dev.fast_trace(s["tree"], s["O"], s["D"], out=s["out"], det_epsilon=s["eps"], reset_depth=True)
    return {"faces_id": out[0], "coords": out[1], "depths": out[2]}


def _deformed(V, seed):
    """This frame's vertices: a sinusoidal displacement of 1% of the extent, as a simulation gives them."""
    g = _gen(seed + 5)
    phase = torch.rand(V.shape[0], 1, generator=g, device="cuda") * 2 * math.pi
    W = V.clone()
    W[:, 2:3] += 0.01 * float((V.amax(0) - V.amin(0)).max()) * torch.sin(phase)
    return W


def _prepare_animate(case, seed):
    V, F = _scene(case, seed)
    n = F.shape[0]
    b = _fast_builder(n, 30)
    keys = torch.empty(n, dtype=torch.int32, device="cuda")
    desc = N.FastBVH(b.nodes.data_ptr(), b.tris.data_ptr(), b.indices.data_ptr(), None, n, 0)
    hb = N.aabox(_hitbox(V))
    N.check(N.lib().rk_fast_build_keyed(dev._stream_ptr(None), F.data_ptr(), V.data_ptr(), n, C.byref(hb), b.mode, 1,
                                        C.byref(desc), b.info.data_ptr(), keys.data_ptr(), b.ws.data_ptr(),
                                        b.ws.numel()), "fast_build_keyed")
    w, h = case["width"], case["height"]
    cam = _camera(case)
    look = -(cam[0][:3] - np.array([0.5, 0.5, 0.1] if case["scene"] == "terrain" else [0, 0, 0], np.float32))
    return {"run": _run_animate, "tree": dev.FastTree(b.nodes, b.tris, b.indices, None, b.info, desc), "F": F,
            "V": _deformed(V, seed), "builder": b, "keys": keys,
            "leaf_faces": F[b.indices.long()].contiguous(), "cam": cam, "w": w, "h": h,
            "look": look / np.linalg.norm(look), "out": dev.new_outputs(w * h),
            "pixels": torch.zeros(w * h, dtype=torch.int32, device="cuda")}


def _run_animate(s):
    b, t = s["builder"], s["tree"]
    N.check(N.lib().rk_fast_refit(dev._stream_ptr(None), s["F"].data_ptr(), s["V"].data_ptr(), s["F"].shape[0], b.mode,
                                  1, C.byref(t.desc), s["keys"].data_ptr(), b.ws.data_ptr(), b.ws.numel()), "fast_refit")
    pixels = dev.render_camera(t, s["cam"], s["w"], s["h"], s["leaf_faces"], s["V"], (0.1, 0.2, 0.3, 1.0), s["look"],
                               pixels=s["pixels"], out=s["out"])
    return {"pixels": pixels, "faces_id": s["out"][0], "coords": s["out"][1], "depths": s["out"][2],
            "nodes": t.nodes, "tris": t.tris.view(torch.int32)}


def _ref_builders(case, n):
    lbvh = sah = None
    if case["tree"] != "sah":
        lbvh = dev.LBVHBuilder(n)
        lbvh.nodes.zero_()  # a tree fills the first of 2n records
    if case["tree"] != "lbvh":
        sah = dev.SAHBuilder(n, 2 * n if case["tree"] == "hybrid" else 0)
    return lbvh, sah


def _prepare_build_ref(case, seed):
    V, F = _scene(case, seed)
    lbvh, sah = _ref_builders(case, F.shape[0])
    return {"run": _run_build_ref, "V": V, "loaded": F, "F": F.clone(), "hitbox": _hitbox(V), "tree": case["tree"],
            "depth": case["depth"], "lbvh": lbvh, "sah": sah}


def _run_build_ref(s):
    F, V, hb = s["F"], s["V"], s["hitbox"]
    F.copy_(s["loaded"])  # a build reorders the faces in place: every pass builds the mesh as it was loaded
    if s["tree"] == "lbvh":
        t = s["lbvh"].build(F, V, hb, s["depth"])
    elif s["tree"] == "sah":
        t = s["sah"].build(F, V, hb)
    else:
        base = s["lbvh"].build(F, V, hb, s["depth"], complete=False)
        base.node_count = int(base.host_info()[N.RK_INFO_NODE_COUNT])  # as the caller of the second build needs it
        t = s["sah"].build(F, V, hb, base)
    return {"nodes": t.nodes, "indices": t.indices, "boxes": t.boxes, "faces": F, "info": t.info[:5]}


def _prepare_trace_ref(case, seed):
    V, F = _scene(case, seed)
    tree = dev.build_lbvh(F, V, _hitbox(V), case["depth"])
    O, D = _rays_of(case, seed)
    return {"run": _run_trace_ref, "tree": tree, "V": V, "O": O, "D": D, "w": case["width"], "h": case["height"],
            "packet": case["packet"], "out": dev.new_outputs(O.shape[0])}


def _run_trace_ref(s):
    fid, uv, dep = s["out"]
    # the buffer's clear, which every frame of the reference starts with
    N.check(N.lib().rk_fill_f32(dev._stream_ptr(None), dep.data_ptr(), dep.numel(), FLT_MAX), "fill")
    dev.trace_ref(s["tree"], s["V"], s["O"], s["D"], s["w"], s["h"], s["packet"], out=s["out"])
    return {"faces_id": fid, "coords": uv, "depths": dep}


def _batch_counts(case):
    """Log-uniform faces and rays of each mesh, a function of the case alone."""
    r = np.random.RandomState(case["meshes"])
    m = case["meshes"]
    faces = (64 * (case["max_faces"] / 64) ** r.random_sample(m)).astype(np.int64)
    rays = (256 * (case["max_rays"] / 256) ** r.random_sample(m)).astype(np.int64)
    return faces, rays


def _batch_input(case, seed):
    """Soups in the unit cube, each with the total area of the 10M-face soup, with scattered rays."""
    faces, rays = _batch_counts(case)
    nf = int(faces.sum())
    scale = torch.from_numpy(np.sqrt(10_000_000 / faces)).cuda().float()
    mesh = torch.repeat_interleave(torch.arange(len(faces), device="cuda"), torch.from_numpy(faces).cuda())
    V, _ = _soup(nf, seed, edge=0.002)
    P = V.reshape(nf, 3, 4)
    mid = P.mean(1, keepdim=True)
    P = mid + (P - mid) * scale[mesh][:, None, None]
    first = torch.from_numpy(np.concatenate([[0], np.cumsum(faces)[:-1]])).cuda()
    local = torch.arange(nf, device="cuda") - first[mesh]
    F = torch.stack([3 * local, 3 * local + 1, 3 * local + 2, torch.zeros_like(local)], 1).int().contiguous()
    lo = torch.full((len(faces), 3), FLT_MAX, device="cuda").scatter_reduce(
        0, mesh[:, None].expand(-1, 3), P[:, :, :3].amin(1), "amin")
    hi = torch.full((len(faces), 3), -FLT_MAX, device="cuda").scatter_reduce(
        0, mesh[:, None].expand(-1, 3), P[:, :, :3].amax(1), "amax")
    boxes = torch.zeros(len(faces), 2, 4, device="cuda")
    boxes[:, 0, :3], boxes[:, 1, :3] = lo, hi
    O, D = _scattered(int(rays.sum()), seed)
    return faces, rays, P.reshape(-1, 4).contiguous(), F, boxes.cpu().numpy(), O, D


def _prepare_batch(case, seed):
    faces, rays, V, F, boxes, O, D = _batch_input(case, seed)
    b = dev.Batch(scenes.batch_table(faces, 3 * faces, rays), F, V, boxes, O, D)
    b.nodes.zero_()  # one record of each mesh is not written
    b.config.ray_order = int(case["sorted"])
    return {"run": _run_batch, "batch": b, "out": dev.new_outputs(O.shape[0])}


def _run_batch(s):
    b, out = s["batch"], s["out"]
    b.build()
    N.check(N.lib().rk_fill_f32(dev._stream_ptr(None), out[2].data_ptr(), out[2].numel(), FLT_MAX), "fill")
    b.trace(out, det_epsilon=0.0)
    return {"nodes": b.nodes, "tris": b.tris.view(torch.int32), "indices": b.indices, "faces_id": out[0],
            "coords": out[1], "depths": out[2]}


def _prepare_serve(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    grids = (32 * (case["max_grid"] / 32) ** np.linspace(0, 1, case["scenes"])).astype(int)
    made = []
    for k, g in enumerate(grids):
        V, F = _terrain(int(g), seed * 64 + k) if k % 2 == 0 else _soup(2 * int(g) ** 2, seed * 64 + k)
        made.append((V.cpu().numpy(), F.cpu().numpy(), k % 2 == 0))
    need = sum(N.lib().rk_server_scene_bytes(V.shape[0], F.shape[0]) + 4096 for V, F, _ in made)
    server = dev.Server(need + (1 << 20), max_faces=max(F.shape[0] for _, F, _ in made),
                        max_pixels=case["max_side"] ** 2)
    ids = [server.add_scene(V, F, z) for V, F, z in made]
    sides = 64 * (case["max_side"] / 64) ** np.random.RandomState(case["requests"]).random_sample(case["requests"])
    asked = []
    for side in sides.astype(int).tolist():
        az, scene = r.uniform(0, 2 * math.pi), int(r.randint(len(ids)))
        mid = np.array([0.5, 0.5, 0.1 if made[scene][2] else 0.5])
        eye = mid + 1.8 * np.array([math.cos(az) * math.cos(math.pi / 6), math.sin(az) * math.cos(math.pi / 6), 0.5])
        cam = N.camera_lookat(eye, mid, math.radians(60.0), side, side, up=[0, 0, 1])
        asked.append((ids[scene], float(r.uniform(0, 10)), cam, side, dev.new_outputs(side * side)))
    return {"run": _run_serve, "server": server, "asked": asked}


def _run_serve(s):
    server = s["server"]
    tickets = [server.submit(scene, time, cam, side, side, out=out) for scene, time, cam, side, out in s["asked"]]
    server.wait_all()
    got = [server.result(t) for t in tickets]
    # a frame's positions depend on when its scene was last rebuilt; its checksum covers the original face ids
    return {"checksums": np.array([g.checksum for g in got], np.uint64).view(np.int64),
            "hits": np.array([g.hits for g in got], np.uint64).view(np.int64),
            "depths": torch.cat([o[2] for *_, o in s["asked"]]), "coords": torch.cat([o[1] for *_, o in s["asked"]])}


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "batch":
        faces, rays = _batch_counts(case)
        nf, nr = float(faces.sum()), float(rays.sum())
        return {"bytes": nf * (16 + 48 + 112 + 4) + nr * 48, "flops": nr * (48 * math.log2(nf / len(faces)) + 53)}
    if kind == "serve":
        k = case["scenes"]
        nf = 2 * sum((32 * (case["max_grid"] / 32) ** x) ** 2 for x in np.linspace(0, 1, k)) / k
        px = (case["max_side"] ** 2 - 64 ** 2) / (2 * math.log(case["max_side"] / 64))
        k = case["requests"]
        return {"bytes": k * (nf * (16 + 2 * 32 + 112) + px * 16),
                "flops": k * (nf * 60 + px * (48 * math.log2(nf) + 53))}
    n, nv = float(_faces(case)), float(_vertices(case))
    mesh = 16 * n + 16 * nv
    if kind == "build_fast":
        return {"bytes": mesh + n * (64 + 48 + 4 + 32), "flops": n * 60}
    if kind == "build_ref":
        return {"bytes": mesh + n * (4 + 32 + 16) + 32 * n / 8, "flops": n * 60}
    rays = float(_ray_count(case))
    per_ray = 48 * math.log2(n) + 53
    if kind == "trace_fast":
        return {"bytes": 112 * n + 48 * rays, "flops": rays * per_ray}
    if kind == "animate":
        return {"bytes": mesh + 8 * n + 112 * n + 20 * rays, "flops": n * 60 + rays * per_ray}
    return {"bytes": mesh + 32 * n / 8 + 48 * rays, "flops": rays * (per_ray + 64 * 53)}


# ---- the same in 64 bits -------------------------------------------------------------

_MOST_TESTS = 4e10  # ray-triangle pairs: about ten seconds


def _closest(O, D, V, F, eps):
    """(u, v), t of each ray's closest triangle by trying all of them; FLT_MAX and (0, 0) where there is none."""
    n = O.shape[0]
    uv = torch.zeros(n, 2, dtype=torch.float64, device="cuda")
    best = torch.full((n,), FLT_MAX, dtype=torch.float64, device="cuda")
    P = V.double()[:, :3][F[:, :3].long()]
    v0, e1, e2 = P[:, 0], P[:, 1] - P[:, 0], P[:, 2] - P[:, 0]
    step = max(1, (1 << 24) // F.shape[0])
    cross = lambda a, b: (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])  # noqa: E731
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1] + a[2] * b[2]  # noqa: E731
    f1, f2 = [e1[:, k] for k in range(3)], [e2[:, k] for k in range(3)]
    for i in range(0, n, step):
        o = [O[i:i + step, k, None].double() for k in range(3)]
        d = [D[i:i + step, k, None].double() for k in range(3)]
        p = cross(d, f2)
        det = dot(f1, p)
        s = [o[k] - v0[:, k] for k in range(3)]
        u = dot(s, p) / det
        q = cross(s, f1)
        v = dot(d, q) / det
        t = dot(f2, q) / det
        ok = (det.abs() >= eps) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0)
        t = torch.where(ok, t, math.inf)
        at = t.argmin(1, keepdim=True)
        t = t.gather(1, at)[:, 0]
        hit = torch.isfinite(t)
        best[i:i + step] = torch.where(hit, t, FLT_MAX)
        uv[i:i + step] = torch.where(hit[:, None], torch.cat([u.gather(1, at), v.gather(1, at)], 1), 0.0)
    return uv, best


def _boxes(V, F):
    P = V.double()[F[:, :3].long()]
    return torch.stack([P.amin(1), P.amax(1)], dim=1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "build_fast":
        V, F = _scene(case, seed)
        return {"nodes": None, "tris": None, "indices": None, "boxes": _boxes(V, F)}
    if kind == "build_ref":
        V, F = _scene(case, seed)
        return {"nodes": None, "indices": None, "boxes": _boxes(V, F), "faces": None, "info": None}
    if kind == "batch":
        faces, rays, V, F, _, O, D = _batch_input(case, seed)
        if float((faces * rays).sum()) > _MOST_TESTS:
            return None
        got, f, r = [], 0, 0
        for nf, nr in zip(faces.tolist(), rays.tolist()):
            got.append(_closest(O[r:r + nr], D[r:r + nr], V[3 * f:3 * (f + nf)], F[f:f + nf], 0.0))
            f, r = f + nf, r + nr
        return {"nodes": None, "tris": None, "indices": None, "faces_id": None,
                "coords": torch.cat([g[0] for g in got]), "depths": torch.cat([g[1] for g in got])}
    if kind == "serve":  # the deformation's phases and axes are the library's own
        return None
    if float(_ray_count(case)) * _faces(case) > _MOST_TESTS:
        return None
    V, F = _scene(case, seed)
    if kind == "animate":
        V = _deformed(V, seed)
    O, D = _rays_of(case, seed)
    uv, t = _closest(O, D, V, F, 0.0 if case["scene"] == "soup" and kind == "trace_fast" else 1e-6)
    got = {"faces_id": None, "coords": uv, "depths": t}
    return {**got, "pixels": None, "nodes": None, "tris": None} if kind == "animate" else got
