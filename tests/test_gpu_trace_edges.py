"""Traces where their launches change. Sorted: at 2^18 faces an XCD takes runs of
512 workgroups (groups of 8 runs, 262144 rays; a remainder in plain order), at 2^20
idle lanes help later. Camera frames, with leaves of one and of several faces. The
closest hit does not depend on any: bit-equal to the trace in ray order. The
reference's per-ray walk: tiles of 16 x 4 rays, whole, cut at an edge, and refused
for too many idle lanes; and its hand-off limits on both sides of 12 rays per face."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("faces", [(1 << 18) - 1, 1 << 18, (1 << 20) - 1, 1 << 20, 1 << 22])
def test_sorted_equals_ray_order(rk, faces):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(faces, seed=faces)
    tree = dev.FastBuilder(faces).build(torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda(), rk.hitbox(V))
    for n in (1, 262143, 262144, 2 * 262144 + 64 * 100 + 1):
        O, D = rk.random_rays(n, seed=n)
        O, D = torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda()
        a = dev.fast_trace_sorted(tree, O, D, det_epsilon=0.0)
        b = dev.fast_trace(tree, O, D, det_epsilon=0.0)  # from 2^22 faces on, late help here too
        c = dev.fast_trace(tree, O, D, det_epsilon=0.0, config=1)
        for x, y, z in zip(a, b, c):
            assert torch.equal(x, y) and torch.equal(x, z)


@pytest.mark.parametrize("leaf_max", [1, 5])
@pytest.mark.parametrize("faces", [(1 << 17) - 1, 1 << 17, 1 << 18, 1 << 20])
def test_sorted_rays_fetch_leaves_apart(rk, faces, leaf_max):
    """Sorted rays on both sides of the face count from which leaves are fetched apart,
    in each kernel that does, with and without a bound of their own, equal to the trace
    in ray order by the plain variant."""
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(faces, seed=faces)
    tree = dev.FastBuilder(faces).build(torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda(),
                                        rk.hitbox(V), leaf_max)
    for n in (1, 63, 70000 + 77):
        O, D = rk.random_rays(n, seed=n)
        o, d = torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda()
        for tmax in (None, 0.25):
            a, b = dev.new_outputs(n, tmax), dev.new_outputs(n, tmax)
            dev.fast_trace_sorted(tree, o, d, a, reset_depth=tmax is None)
            dev.fast_trace(tree, o, d, b, config=1, reset_depth=tmax is None)
            for x, y in zip(a, b):
                assert torch.equal(x, y)


@pytest.mark.parametrize("w,h", [(1, 1), (641, 512)])
@pytest.mark.parametrize("leaf_max", [1, 5, 16])
def test_camera_equals_rays(rk, w, h, leaf_max):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(20000, seed=w)
    tree = dev.FastBuilder(20000).build(torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda(),
                                        rk.hitbox(V), leaf_max)
    cam = rk.camera_lookat([0.5, -1.5, 0.9], [0.5, 0.5, 0.5], 0.8, w, h, up=[0, 0, 1])
    O, D = rk.primary_rays_host(cam, w, h)
    a = dev.fast_trace_camera(tree, cam, w, h, det_epsilon=0.0)
    b = dev.fast_trace(tree, torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda(), det_epsilon=0.0)
    hit = b[2] < torch.finfo(torch.float32).max
    assert torch.equal(a[2], b[2]) and (w == 1 or bool(hit.any()))
    assert torch.equal(a[0][hit], b[0][hit]) and torch.equal(a[1][hit], b[1][hit])


@pytest.mark.parametrize("w,h", [(64, 48), (120, 64), (128, 50), (67, 50), (16, 4), (15, 4), (1000, 1), (1, 1000)])
def test_reference_rays_in_tiles(rk, ora, w, h):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(3000, seed=w, mu=float(np.log(0.1)))
    hb = rk.hitbox(V)
    ref = ora.build_lbvh_ref(F, V, hb, 12, True)
    Ft, Vt = torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda()
    tree = dev.build_lbvh(Ft, Vt, hb, 12, True)
    O, D = rk.random_rays(w * h, seed=h)
    of, ouv, od, _ = ora.trace_ref_ray(ref.nodes, ref.faces, V, O, D)
    out = dev.trace_ref(tree, Vt, torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda(), w, h, False)
    got = [t.cpu().numpy() for t in out]
    np.testing.assert_array_equal(got[0].view(np.uint32), of)
    np.testing.assert_array_equal(got[1], ouv)
    np.testing.assert_array_equal(got[2], od)


@pytest.mark.parametrize("coherency", [False, True])
@pytest.mark.parametrize("faces,w,h", [(16384, 512, 384), (16385, 512, 384), (16384, 512, 383), (5461, 256, 256),
                                       (5462, 256, 256)])
def test_reference_handoff_limit_by_rays_per_face(rk, faces, w, h, coherency):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(faces, seed=faces)
    hb = rk.hitbox(V)
    Ft, Vt = torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda()
    tree = dev.build_lbvh(Ft, Vt, hb, 12, True)
    O, D = rk.random_rays(w * h, seed=h)
    O, D = torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda()
    a = dev.trace_ref(tree, Vt, O, D, w, h, coherency)
    try:
        dev.set_ref_handoff(0xFFFFFFFF, 0xFFFFFFFF)  # no second passes
        b = dev.trace_ref(tree, Vt, O, D, w, h, coherency)
    finally:
        dev.set_ref_handoff()
    for x, y in zip(a, b):
        assert torch.equal(x, y)


def _eight_leaves(ora, leaf):
    """Eight leaves of 'leaf' scattered faces each at the corners of a cube, under a
    tree of three levels."""
    rng = np.random.default_rng(leaf)
    corner = np.array([[x, y, z] for x in (.25, .75) for y in (.25, .75) for z in (.25, .75)])
    P = corner[:, None, None] + rng.normal(0, .05, (8, leaf, 1, 3)) + rng.normal(0, .04, (8, leaf, 3, 3))
    V, F = np.zeros((24 * leaf, 4), np.float32), np.zeros((8 * leaf, 4), np.uint32)
    V[:, :3] = P.reshape(-1, 3)
    F[:, :3] = np.arange(24 * leaf, dtype=np.uint32).reshape(-1, 3)
    nodes = np.zeros(15, ora.NODE_DTYPE)
    for k in range(14, -1, -1):  # heap order: children 2k + 1, 2k + 2
        if k >= 7:
            T = V[3 * leaf * (k - 7):3 * leaf * (k - 6), :3]
            nodes[k] = (1 | leaf << 1, leaf * (k - 7), T.min(0), T.max(0))
        else:
            a, b = nodes[2 * k + 1], nodes[2 * k + 2]
            axis = 0 if k == 0 else (1 if k < 3 else 2)
            nodes[k] = (axis << 1, 2 * k + 1, np.minimum(a["bmin"], b["bmin"]), np.maximum(a["bmax"], b["bmax"]))
    return V, F, nodes


def _trace(dev, nodes, V, F, O, D, w, h, packet):
    import torch
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    tree = dev.RefTree(t(F.view(np.int32)), None, None, t(nodes.view(np.int32).reshape(-1, 8)), None, len(nodes))
    return [x.cpu().numpy() for x in dev.trace_ref(tree, t(V), t(O), t(D), w, h, packet)]


@pytest.mark.parametrize("leaf", [1, 4, 5, 16, 17, 63, 64, 65, 200])
@pytest.mark.parametrize("w,h", [(256, 255), (256, 256), (331, 200), (300, 222)])
def test_reference_rays_of_small_and_large_frames(rk, ora, w, h, leaf):
    """Frames on both sides of 2^16 rays, in rows and in tiles (whole, cut at the
    right, at the bottom), where the leaves' faces are tested with and without their
    bounds, by a lane and by the wave."""
    from cudart_amd import device as dev
    V, F, nodes = _eight_leaves(ora, leaf)
    cam = rk.camera_lookat([.7, .35, 2.2], [.5, .5, .5], .7, w, h, up=[0, 1, 0])
    O, D = rk.primary_rays_host(cam, w, h)
    of, ouv, od, _ = ora.trace_ref_ray(nodes, F, V, O, D)
    assert 0.001 < (od < np.finfo(np.float32).max).mean() < 0.9
    got = _trace(dev, nodes, V, F, O, D, w, h, False)
    np.testing.assert_array_equal(got[0].view(np.uint32), of)
    np.testing.assert_array_equal(got[1], ouv)
    np.testing.assert_array_equal(got[2], od)


@pytest.mark.parametrize("leaf", [1, 2, 3, 15, 16, 17, 96, 97])
@pytest.mark.parametrize("first_pass", [True, False])
def test_packet_leaf_sizes(rk, ora, leaf, first_pass):
    """Leaves whose faces come through the scalar cache, without and with their
    bounds, in the first pass and in the second."""
    from cudart_amd import device as dev
    V, F, nodes = _eight_leaves(ora, leaf)
    w, h = 131, 89
    cam = rk.camera_lookat([.7, .35, 2.2], [.5, .5, .5], .7, w, h, up=[0, 1, 0])
    O, D = rk.primary_rays_host(cam, w, h)
    of, ouv, od, _ = ora.trace_ref_packet(nodes, F, V, O, D, w, h)
    assert 0.001 < (od < np.finfo(np.float32).max).mean() < 0.9
    try:
        dev.set_ref_handoff(packet_faces=0xFFFFFFFF if first_pass else 0)
        got = _trace(dev, nodes, V, F, O, D, w, h, True)
    finally:
        dev.set_ref_handoff()
    np.testing.assert_array_equal(got[0].view(np.uint32), of)
    np.testing.assert_array_equal(got[1], ouv)
    np.testing.assert_array_equal(got[2], od)


@pytest.mark.parametrize("every", [True, False])
def test_more_forced_packets_than_the_split_takes(rk, ora, every):
    """A frame of 1,225 packets, each with a ray (or all its rays) whose direction has
    a component of 0: the split takes 1,024 of them."""
    from cudart_amd import device as dev
    V, F, nodes = _eight_leaves(ora, 16)
    w, h = 560, 420
    cam = rk.camera_lookat([2.2, .35, .6], [.5, .5, .5], .6, w, h, up=[0, 1, 0])
    O, D = rk.primary_rays_host(cam, w, h)
    O = O.reshape(h, w, 4).copy()
    D = D.reshape(h, w, 4).copy()
    pick = np.s_[:, :] if every else np.s_[2::12, 3::16]
    D[pick][..., 2] = 0
    O[pick][..., 2] = np.linspace(.1, .9, O[pick].shape[1], dtype=np.float32)
    O, D = O.reshape(-1, 4), D.reshape(-1, 4)
    of, ouv, od, _ = ora.trace_ref_packet(nodes, F, V, O, D, w, h)
    assert 0.01 < (od < np.finfo(np.float32).max).mean() < 0.9
    got = _trace(dev, nodes, V, F, O, D, w, h, True)
    np.testing.assert_array_equal(got[0].view(np.uint32), of)
    np.testing.assert_array_equal(got[1], ouv)
    np.testing.assert_array_equal(got[2], od)


@pytest.mark.parametrize("packet", [True, False])
def test_split_walks_past_their_hit_lists(rk, ora, packet):
    """256 subtrees of two faces, layers one behind the other: rays that walk every
    subtree hit most of them, more than the lists hold (32 entries per ray, 2 per
    packet's ray, on average)."""
    from cudart_amd import device as dev
    rng = np.random.default_rng(8)
    n, w, h = 256, 64, 48
    P = np.zeros((n, 2, 3, 3))
    P[..., 0] = np.linspace(0, 1, n)[:, None, None] + rng.uniform(0, 1e-3, (n, 2, 3))
    P[:, 0, :, 1:] = [(-.2, -.2), (1.2, -.2), (-.2, 1.2)]
    P[:, 1, :, 1:] = [(1.2, 1.2), (-.2, 1.2), (1.2, -.2)]
    P[..., 1:] += rng.normal(0, .02, (n, 2, 3, 2))
    order = rng.permutation(n)  # the nearest layer in no particular subtree
    V, F = np.zeros((6 * n, 4), np.float32), np.zeros((2 * n, 4), np.uint32)
    V[:, :3] = P[order].reshape(-1, 3)
    F[:, :3] = np.arange(6 * n, dtype=np.uint32).reshape(-1, 3)
    nodes = np.zeros(2 * n - 1, ora.NODE_DTYPE)
    for k in range(2 * n - 2, -1, -1):
        if k >= n - 1:
            T = V[6 * (k - n + 1):6 * (k - n + 2), :3]
            nodes[k] = (1 | 2 << 1, 2 * (k - n + 1), T.min(0), T.max(0))
        else:
            a, b = nodes[2 * k + 1], nodes[2 * k + 2]
            nodes[k] = ((k % 3) << 1, 2 * k + 1, np.minimum(a["bmin"], b["bmin"]), np.maximum(a["bmax"], b["bmax"]))
    O, D = np.zeros((w * h, 4), np.float32), np.zeros((w * h, 4), np.float32)
    O[:, 0] = -1
    O[:, 1:3] = rng.uniform(0, 1, (w * h, 2))
    D[:, 0] = 1
    D[:, 1] = rng.normal(0, .05, w * h)
    hits = 0
    for k in range(n - 1, 2 * n - 1):
        hits += int((ora.trace_ref_ray(nodes[k:k + 1], F, V, O, D)[2] < np.finfo(np.float32).max).sum())
    assert hits > 2 * 32 * w * h
    if packet:
        of, ouv, od, _ = ora.trace_ref_packet(nodes, F, V, O, D, w, h)
    else:
        of, ouv, od, _ = ora.trace_ref_ray(nodes, F, V, O, D)
    got = _trace(dev, nodes, V, F, O, D, w, h, packet)
    np.testing.assert_array_equal(got[0].view(np.uint32), of)
    np.testing.assert_array_equal(got[1], ouv)
    np.testing.assert_array_equal(got[2], od)
