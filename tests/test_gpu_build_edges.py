"""The sort and the hierarchy pass at the sizes where their launches change: tiles
and groups of tiles of the sort, the one-workgroup sort, runs and groups of runs of
the hierarchy; the reference topology where a level or the split lists stop
fitting in LDS; the SAH build where its items change hands."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SORT_SIZES = [2, 513, 2048, 2049, 4096, 4097, 16 * 2048, 16 * 2048 + 1, (1 << 19) - 1, 1 << 19, (1 << 21) - 1, 1 << 21]


@pytest.mark.parametrize("n", SORT_SIZES)
def test_sorts_at_tile_edges(n):
    """32-bit and 64-bit pairs with many equal keys, odd and even numbers of
    passes, against numpy's stable sort."""
    import torch

    from cudart_amd import device as dev
    rng = np.random.default_rng(n)
    for bits in (8, 24, 32, 40, 64):
        wide = bits > 32
        k = rng.integers(0, 1 << min(bits, 63), n, dtype=np.uint64) & rng.integers(0, 1 << min(bits, 63), n, dtype=np.uint64)
        k = k if wide else k.astype(np.uint32)
        v = np.arange(n, dtype=np.uint32)[::-1].copy()
        kt = torch.from_numpy(k.view(np.int64 if wide else np.int32).copy()).cuda()
        vt = torch.from_numpy(v.view(np.int32)).cuda()
        if wide:
            dev.sort_pairs_u64(kt, vt, bits)
        elif n > 32768 or n <= 512:  # between, the reference's bitonic chunks order equal keys
            dev.sort_general(kt, vt, bits)
        else:
            dev.sort_values(kt, bits)
        order = np.argsort(k, kind="stable")
        np.testing.assert_array_equal(kt.cpu().numpy().view(k.dtype), k[order])
        if wide or n > 32768 or n <= 512:
            np.testing.assert_array_equal(vt.cpu().numpy().view(np.uint32), v[order])


def _split(keys, i):
    x = int(keys[i]) ^ int(keys[i + 1])
    return (x | 1 << 63) if x else (i ^ (i + 1))


def _expected(keys):
    """{record: (left ref, right ref, left count, right count)} of the binary radix
    tree over sorted keys, one face per leaf, from a stack of the splits' keys."""
    n = len(keys)
    up = [_split(keys, i) for i in range(n - 1)]
    first = [0] * (n - 1)
    last = [n - 1] * (n - 1)
    stack = []  # each split's range ends at the nearest larger split on either side
    for i, k in enumerate(up):
        while stack and up[stack[-1]] < k:
            last[stack.pop()] = i
        first[i] = stack[-1] + 1 if stack else 0
        stack.append(i)

    def record(l, r):
        if l == r:
            return 0x80000000 | l << 4
        if (l, r) == (0, n - 1):
            return 0
        left = l == 0 or (r + 1 < n and up[r] < up[l - 1])
        return r if left else l
    return {record(first[p], last[p]): (record(first[p], p), record(p + 1, last[p]), p - first[p] + 1, last[p] - p)
            for p in range(n - 1)}


@pytest.mark.parametrize("n", [2, 3, 511, 512, 513, 1024, 1025, 40 * 512, 40 * 512 + 1, 64 * 512, 64 * 512 + 1, 70001])
@pytest.mark.parametrize("kind", ["soup30", "soup63", "equal", "chain"])
def test_hierarchy_topology_at_run_edges(rk, n, kind):
    """Every record of the tree against the tree computed from the sorted keys:
    random faces, all faces with one key, and keys whose splits form a chain that
    leaves over as many subtrees per run as the key length allows."""
    import torch
    V, F = rk.soup(n, seed=n)
    if kind == "equal":
        F = np.repeat(F[:1], n, axis=0)
    elif kind == "chain":  # centroids halve towards one corner, over and over
        c = np.float32(0.5) ** np.arange(n, dtype=np.float32).clip(0, 20)
        V = V.reshape(n, 3, 4)
        V[:, :, :3] = c[:, None, None] * np.float32(1.0)
        V = np.ascontiguousarray(V.reshape(-1, 4))
    hb = rk.hitbox(V)
    mode = rk.RK_MORTON_63 if kind == "soup63" else rk.RK_MORTON_30
    L = rk.lib()
    Ft, Vt = torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda()
    nodes = torch.zeros((n, 16), dtype=torch.int32, device="cuda")
    tris = torch.zeros((n, 12), dtype=torch.float32, device="cuda")
    order = torch.zeros(n, dtype=torch.int32, device="cuda")
    keys = torch.zeros(n, dtype=torch.int64 if kind == "soup63" else torch.int32, device="cuda")
    info = torch.zeros(8, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.rk_fast_build_workspace_size(n, mode), dtype=torch.uint8, device="cuda")
    desc = rk.FastBVH(nodes.data_ptr(), tris.data_ptr(), order.data_ptr(), None, n, 0)
    box = rk.aabox(hb)
    rk.check(L.rk_fast_build_keyed(None, Ft.data_ptr(), Vt.data_ptr(), n, C.byref(box), mode, 1, C.byref(desc),
                                   info.data_ptr(), keys.data_ptr(), ws.data_ptr(), ws.numel()), "build")
    torch.cuda.synchronize()
    k = keys.cpu().numpy().view(np.uint64 if kind == "soup63" else np.uint32)
    assert (np.diff(k.astype(np.float64)) >= 0).all()
    np.testing.assert_array_equal(np.sort(order.cpu().numpy()), np.arange(n))
    got = nodes.cpu().numpy().view(np.uint32)
    boxes = got[:, :12].copy().view(np.float32)
    expect = _expected(k)
    idx = np.fromiter(expect, np.int64)
    np.testing.assert_array_equal(got[idx, 12:], np.array(list(expect.values()), np.uint32))
    # the root's two boxes hold every vertex
    lo = np.minimum(boxes[0, [0, 2, 8]], boxes[0, [4, 6, 10]])
    hi = np.maximum(boxes[0, [1, 3, 9]], boxes[0, [5, 7, 11]])
    P = V[F[:, :3]].reshape(-1, 4)[:, :3]
    assert (lo <= P.min(0)).all() and (hi >= P.max(0)).all()


# faces: groups of 512 split bits; 16384 splits and levels of 3072 and 5120
# records (LDS). "same": one code, so every split is a median's, by levels of 2^L.
@pytest.mark.parametrize("n,depth,complete,same", [
    (1, 12, True, False), (2, 31, True, False), (225, 12, True, True), (511, 31, True, False), (512, 31, True, False),
    (513, 31, False, False), (16385, 31, True, False), (16386, 31, True, False), (60001, 31, True, False),
    (150000, 31, True, False), (150000, 14, False, False), (1200000, 12, True, True)])
def test_reference_topology_at_lds_edges(rk, ora, n, depth, complete, same):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(n, seed=n)
    if same:
        F = np.repeat(F[:1], n, axis=0)
    hb = rk.hitbox(V)
    ref = ora.build_lbvh_ref(F, V, hb, depth, complete)
    Ft = torch.from_numpy(F.view(np.int32).copy()).cuda()
    tree = dev.build_lbvh(Ft, torch.from_numpy(V).cuda(), hb, depth, complete)
    info = tree.host_info()
    m = int(info[rk.RK_INFO_NODE_COUNT])
    assert m == ref.node_count and int(info[rk.RK_INFO_REAL_DEPTH]) == ref.real_depth
    assert int(info[rk.RK_INFO_FLAGS]) & 0xFF == ref.flags
    np.testing.assert_array_equal(tree.indices.cpu().numpy().view(np.uint32), ref.indices)
    np.testing.assert_array_equal(Ft.cpu().numpy().view(np.uint32), ref.faces)
    nodes = tree.nodes.cpu().numpy().view(np.uint32)[:m].copy().view(ora.NODE_DTYPE).reshape(m)
    for name in ("w0", "w1", "bmin", "bmax"):  # boxes as floats: -0 == +0
        assert np.array_equal(nodes[name], ref.nodes[name]), name


def _chain(per):
    """Faces at distances 2^-60 to 2^60 along each axis, 'per' to an octave: a SAH
    tree of more than 64 levels."""
    rng = np.random.default_rng(per)
    c = np.zeros((3, 120, per, 3), np.float32)
    for a in range(3):
        c[a, :, :, a] = 2.0 ** np.arange(-60, 60)[:, None] * rng.uniform(1, 2, (120, per))
    c = c.reshape(-1, 3)
    d = np.abs(c).max(1, keepdims=True) * np.float32(2.0 ** -10)
    corners = np.stack([c, c + d * np.array([1, 0, .5], np.float32), c + d * np.array([0, 1, .5], np.float32)], 1)
    n = len(c)
    V, F = np.zeros((3 * n, 4), np.float32), np.zeros((n, 4), np.uint32)
    V[:, :3] = corners.reshape(-1, 3)
    F[:, :3] = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    return V, F


# items of 16, 128, 256, 512 and 1024 faces; chunks of 1024; levels of more than 1024 items
@pytest.mark.parametrize("scene", [1, 16, 17, 127, 129, 256, 257, 511, 513, 1024, 1025, 2048, 2049, 70000, "chain4",
                                   "chain40"])
def test_sah_at_item_edges(rk, ora, scene):
    import torch

    from cudart_amd import device as dev
    V, F = _chain(int(scene[5:])) if isinstance(scene, str) else rk.soup(scene, seed=scene)
    hb = rk.hitbox(V)
    boxes, idx = ora.calc_boxes(F, V)
    nodes, order, flags = ora.build_sah(boxes, idx, hb)
    Ft = torch.from_numpy(F.view(np.int32).copy()).cuda()
    tree = dev.build_sah(Ft, torch.from_numpy(V).cuda(), hb)
    _compare_sah(rk, ora, F, Ft, tree, nodes, order, flags)


@pytest.mark.parametrize("n,depth,complete", [(60000, 31, True), (60000, 8, False), (3000, 3, False), (17, 0, False)])
def test_hybrid_at_item_edges(rk, ora, n, depth, complete):
    """Thousands of small leaves, a few of thousands of faces, and one."""
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(n, seed=n + depth)
    hb = rk.hitbox(V)
    ref = ora.build_lbvh_ref(F, V, hb, depth, False)
    if complete:
        ref = ora.build_lbvh_ref(F, V, hb, depth, True)
        F = ref.faces
    boxes, idx = (ref.boxes, ref.indices) if not complete else ora.calc_boxes(F, V)
    nodes, order, flags = ora.build_sah(boxes, idx, hb, ref.nodes, ref.node_count)
    Ft, Vt = torch.from_numpy(F.view(np.int32).copy()).cuda(), torch.from_numpy(V).cuda()
    lb = dev.build_lbvh(Ft, Vt, hb, depth, complete)
    if complete:  # its faces are in tree order: boxes and ids of those
        assert lb.node_count == ref.node_count
        Ft = torch.from_numpy(F.view(np.int32).copy()).cuda()
        lb.boxes.copy_(torch.from_numpy(boxes.reshape(lb.boxes.shape)))
        lb.indices.copy_(torch.from_numpy(idx.view(np.int32).reshape(lb.indices.shape)))
    tree = dev.build_sah(Ft, Vt, hb, lbvh=lb)
    _compare_sah(rk, ora, F, Ft, tree, nodes, order, flags)


def _compare_sah(rk, ora, F, Ft, tree, nodes, order, flags):
    m = tree.node_count
    assert m == nodes.shape[0] and int(tree.host_info()[rk.RK_INFO_FLAGS]) == flags
    np.testing.assert_array_equal(tree.indices.cpu().numpy().view(np.uint32), order)
    np.testing.assert_array_equal(Ft.cpu().numpy().view(np.uint32), F[order])
    got = tree.nodes.cpu().numpy().view(np.uint32)[:m].copy().view(ora.NODE_DTYPE).reshape(m)
    for name in ("w0", "w1", "bmin", "bmax"):
        assert np.array_equal(got[name], nodes[name]), name


@pytest.mark.parametrize("n", [1, 16, 1000, 1024])
def test_sah_small_root_keeps_no_bounds(rk, n):
    """A root that goes straight to the small items has no room for centroid bounds
    in the workspace: theirs (as ordered ints, the bits of a positive float) are
    nowhere in it, whatever it held before."""
    import torch
    V, F = rk.soup(n, seed=n, lo=1.0, hi=2.0)
    hb = rk.aabox(rk.hitbox(V))
    L = rk.lib()
    Ft, Vt = torch.from_numpy(F.view(np.int32).copy()).cuda(), torch.from_numpy(V).cuda()
    boxes = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    ids = torch.zeros(n, dtype=torch.int32, device="cuda")
    nodes = torch.zeros((2 * n, 8), dtype=torch.int32, device="cuda")
    info = torch.zeros(8, dtype=torch.int32, device="cuda")
    ws = torch.full((L.rk_build_sah_workspace_size(n, 0) // 4,), 0x7FFFFFFF, dtype=torch.int32, device="cuda")
    rk.check(L.rk_build_sah(None, Ft.data_ptr(), Vt.data_ptr(), n, C.byref(hb), boxes.data_ptr(), ids.data_ptr(),
                            nodes.data_ptr(), 0, 2 * n, info.data_ptr(), ws.data_ptr(), 4 * ws.numel()), "sah")
    torch.cuda.synchronize()
    T = V[F[:, :3], :3]
    low = ((T.min(1) + T.max(1)) * np.float32(0.5)).min(0)
    assert (low > 0).all() and not np.isin(low.view(np.int32), ws.cpu().numpy()).any()


def _comb(n):
    """n faces in parallel planes, so large that every split of them costs the same:
    the SAH takes the last one, which holds the last face alone (the distances from
    the first are those whose 31 / d * d does not round below 31). A face per level,
    down to a leaf of 223: internal items on levels 0 to n - 224."""
    d = np.arange(1, 4 * n, dtype=np.float32)
    d = d[np.float32(31) / d * d >= 31][:n - 1]
    assert len(d) == n - 1
    V, F = np.zeros((n, 3, 4), np.float32), np.zeros((n, 4), np.uint32)
    V[1:, :, 0] = d[:, None]
    V[:, 1, 1] = V[:, 2, 2] = 1e15
    F[:, :3] = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    return V.reshape(-1, 4), F


def test_sah_at_the_depth_limit(rk, ora):
    """The deepest tree the build takes, 4096 levels with internal items."""
    import torch

    from cudart_amd import device as dev
    V, F = _comb(4096 + 223)
    hb = rk.hitbox(V)
    boxes, idx = ora.calc_boxes(F, V)
    nodes, order, flags = ora.build_sah(boxes, idx, hb)
    assert nodes.shape[0] == 2 * 4096 + 1
    Ft = torch.from_numpy(F.view(np.int32).copy()).cuda()
    tree = dev.build_sah(Ft, torch.from_numpy(V).cuda(), hb)
    _compare_sah(rk, ora, F, Ft, tree, nodes, order, flags)


@pytest.mark.parametrize("n", [4096 + 224, 4096 + 1024 + 2])  # met by a small item, by a large one
def test_sah_past_the_depth_limit_leaves_the_faces(rk, n):
    import torch

    from cudart_amd import device as dev
    V, F = _comb(n)
    F = F[np.random.default_rng(n).permutation(n)]
    Ft = torch.from_numpy(F.view(np.int32).copy()).cuda()
    with pytest.raises(rk.RkError, match=r"\(3\)"):
        dev.build_sah(Ft, torch.from_numpy(V).cuda(), rk.hitbox(V))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(Ft.cpu().numpy().view(np.uint32), F)


def test_hybrid_without_leaves_counts_the_nodes(rk):
    """Existing nodes that hold no leaf leave nothing to refine: the node count is
    theirs, and the faces follow the indices."""
    import torch
    n, existing = 40, 3
    V, F = rk.soup(n, seed=n)
    hb = rk.aabox(rk.hitbox(V))
    L = rk.lib()
    order = np.random.default_rng(n).permutation(n).astype(np.uint32)
    Ft, Vt = torch.from_numpy(F.view(np.int32).copy()).cuda(), torch.from_numpy(V).cuda()
    boxes = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    ids = torch.from_numpy(order.view(np.int32)).cuda()
    nodes = torch.zeros((existing + 2 * n, 8), dtype=torch.int32, device="cuda")
    info = torch.full((8,), -1, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.rk_build_sah_workspace_size(n, existing), dtype=torch.uint8, device="cuda")
    rk.check(L.rk_build_sah(None, Ft.data_ptr(), Vt.data_ptr(), n, C.byref(hb), boxes.data_ptr(), ids.data_ptr(),
                            nodes.data_ptr(), existing, existing + 2 * n, info.data_ptr(), ws.data_ptr(),
                            ws.numel()), "sah")
    torch.cuda.synchronize()
    assert info.cpu().tolist()[:3] == [existing, 0, 0] and not nodes.any()
    np.testing.assert_array_equal(Ft.cpu().numpy().view(np.uint32), F[order])


def test_sah_lets_no_exception_out():
    """The build with no C++ heap at hand (tests/cpp/no_heap.cpp)."""
    exe = Path(__file__).resolve().parent / "cpp" / "_build" / "no_heap"
    assert exe.exists(), "build() compiles tests/cpp first"
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "status 0" in r.stdout, r.stdout + r.stderr
