"""Sorted traces where their launches change: at 2^18 faces an XCD takes runs of
512 workgroups (groups of 8 runs, 262144 rays; a remainder in plain order), at 2^20
idle lanes help later. The closest hit does not depend on either: bit-equal to the
trace in ray order."""
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
