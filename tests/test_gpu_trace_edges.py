"""Traces where their launches change. Sorted: at 2^18 faces an XCD takes runs of
512 workgroups (groups of 8 runs, 262144 rays; a remainder in plain order), at 2^20
idle lanes help later. Camera frames: at 327680 pixels. The closest hit does not
depend on any: bit-equal to the trace in ray order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("faces", [(1 << 18) - 1, 1 << 18, (1 << 20) - 1, 1 << 20])
def test_sorted_equals_ray_order(rk, faces):
    import torch

    from cudart_amd import device as dev
    V, F = rk.soup(faces, seed=faces)
    tree = dev.FastBuilder(faces).build(torch.from_numpy(F.view(np.int32)).cuda(), torch.from_numpy(V).cuda(), rk.hitbox(V))
    for n in (1, 262143, 262144, 2 * 262144 + 64 * 100 + 1):
        O, D = rk.random_rays(n, seed=n)
        O, D = torch.from_numpy(O).cuda(), torch.from_numpy(D).cuda()
        a = dev.fast_trace_sorted(tree, O, D, det_epsilon=0.0)
        b = dev.fast_trace(tree, O, D, det_epsilon=0.0)
        for x, y in zip(a, b):
            assert torch.equal(x, y)


@pytest.mark.parametrize("w,h", [(1, 1), (640, 512), (641, 512)])
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
