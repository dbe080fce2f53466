"""The least workspace of the sorts and of the fast and batch builds: one byte less is
refused and touches nothing, and with exactly that the results are right, whichever
kernels a size goes to."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ERROR_WORKSPACE = 4


def _up(x):
    return (x + 255) // 256 * 256


def _least_sort(n, key_bytes, passes, pairs):
    """A word, a row of 256 counts per pass and a row per pass and tile, then the other
    halves of the keys and the values."""
    tile = 4096 if n < 1 << 21 else 8192
    T = (n + tile - 1) // tile
    head = _up(4 * (1 + 256 * passes + 256 * passes * T))
    return head + (_up(key_bytes * n) + 4 * n if pairs else key_bytes * n)


# one workgroup up to 4096 keys; tiles of 2048, 4096 (from 2^19) and 8192 keys (from 2^21)
@pytest.mark.parametrize("n", [2, 4096, 4097, 70001, 1 << 19, (1 << 21) - 1, 1 << 21])
@pytest.mark.parametrize("bits", [8, 16, 64])
def test_sort_least_workspace(rk, n, bits):
    import torch
    rng = np.random.default_rng(n + bits)
    k = rng.integers(0, 1 << min(bits, 63), n, dtype=np.uint64)
    v = rng.permutation(n).astype(np.uint32)
    kt, vt = torch.from_numpy(k.view(np.int64)).cuda(), torch.from_numpy(v.view(np.int32)).cuda()
    need = _least_sort(n, 8, bits // 8, True)
    assert need <= rk.lib().rk_sort_workspace_size(n, 8)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    sort = lambda size: rk.lib().rk_radix_sort_pairs_u64(None, kt.data_ptr(), vt.data_ptr(), n, bits, ws.data_ptr(),
                                                         size)
    assert sort(need - 1) == ERROR_WORKSPACE
    torch.cuda.synchronize()
    np.testing.assert_array_equal(kt.cpu().numpy().view(np.uint64), k)
    assert not ws.any()
    assert sort(need) == 0
    torch.cuda.synchronize()
    order = np.argsort(k, kind="stable")
    np.testing.assert_array_equal(kt.cpu().numpy().view(np.uint64), k[order])
    np.testing.assert_array_equal(vt.cpu().numpy().view(np.uint32), v[order])
    assert not ws[need:].any() and not ws[:4].any()


@pytest.mark.parametrize("n", [513, 4096, 40000, 600000])
def test_value_sort_least_workspace(rk, n):
    import torch
    k = np.random.default_rng(n).integers(0, 1 << 8, n, dtype=np.uint64).astype(np.uint32)
    kt = torch.from_numpy(k.view(np.int32)).cuda()
    need = _least_sort(n, 4, 4 if n <= 8192 else 1, False)  # small sorts compare whole values
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    sort = lambda size: rk.lib().rk_radix_sort(None, kt.data_ptr(), n, 8, ws.data_ptr(), size)
    assert sort(need - 1) == ERROR_WORKSPACE and sort(need) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(kt.cpu().numpy().view(np.uint32), np.sort(k))


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("n", [1, 300, 4097, 70001])
def test_fast_build_and_refit_least_workspace(rk, n, mode):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(n, seed=n)
    hb = rk.hitbox(V)
    box = rk.aabox(hb)
    L = rk.lib()
    Ft, Vt = torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda()
    want = dev.FastBuilder(n, mode).build(Ft, Vt, hb)
    nodes = torch.zeros((n, 16), dtype=torch.int32, device="cuda")
    tris = torch.zeros((n, 12), dtype=torch.float32, device="cuda")
    order = torch.zeros(n, dtype=torch.int32, device="cuda")
    keys = torch.zeros(n, dtype=torch.int64, device="cuda")
    info = torch.zeros(8, dtype=torch.int32, device="cuda")
    desc = rk.FastBVH(nodes.data_ptr(), tris.data_ptr(), order.data_ptr(), None, n, 0)
    need = L.rk_fast_build_workspace_size(n, mode) - 4096
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    build = lambda size: L.rk_fast_build_keyed(None, Ft.data_ptr(), Vt.data_ptr(), n, C.byref(box), mode, 1,
                                               C.byref(desc), info.data_ptr(), keys.data_ptr(), ws.data_ptr(), size)
    assert build(need - 1) == ERROR_WORKSPACE
    torch.cuda.synchronize()
    assert not nodes.any() and not order.any()
    assert build(need) == 0
    torch.cuda.synchronize()
    assert torch.equal(order, want.indices[:n]) and torch.equal(tris.view(torch.int32), want.tris[:n].view(torch.int32))
    first = nodes.clone()
    need = 2 * _up(4 * n) + _up(48 * n) + 4 * ((n + 511) // 512)
    refit = lambda size: L.rk_fast_refit(None, Ft.data_ptr(), Vt.data_ptr(), n, mode, 1, C.byref(desc),
                                         keys.data_ptr(), ws.data_ptr(), size)
    nodes.zero_()
    assert refit(need - 1) == ERROR_WORKSPACE
    torch.cuda.synchronize()
    assert not nodes.any()
    assert refit(need) == 0
    torch.cuda.synchronize()
    assert torch.equal(nodes, first)


def test_batch_build_least_workspace(rk):
    import torch

    from cudart_amd import device as dev
    counts = [1, 300, 4000, 700]
    meshes = [rk.soup(c, seed=c) for c in counts]
    V, F = np.concatenate([m[0] for m in meshes]), np.concatenate([m[1] for m in meshes])
    table = np.zeros(len(counts), rk.BATCH_MESH_DTYPE)
    table["face_count"], table["vertex_count"], table["ray_count"] = counts, [3 * c for c in counts], 1
    for a in ("face", "vertex", "ray"):
        table[a + "_offset"] = np.concatenate([[0], np.cumsum(table[a + "_count"])[:-1]])
    O, D = rk.random_rays(len(counts), seed=1)
    t = lambda a: torch.from_numpy(a).cuda()
    b = dev.Batch(table, t(F.view(np.int32)), t(V), np.stack([rk.hitbox(m[0]) for m in meshes]), t(O), t(D))
    b.nodes.zero_()
    b.build()
    want = b.nodes.clone(), b.tris.view(torch.int32).clone(), b.indices.clone()
    need = rk.lib().rk_batch_build_workspace_size(len(counts), int(F.shape[0])) - 4096
    b.nodes.zero_()
    b.build_bytes = need - 1
    with pytest.raises(rk.RkError, match=r"\(4\)"):
        b.build()
    torch.cuda.synchronize()
    assert not b.nodes.any()
    b.build_bytes = need
    b.build()
    torch.cuda.synchronize()
    for got, w in zip((b.nodes, b.tris.view(torch.int32), b.indices), want):
        assert torch.equal(got, w)
