"""The shade adjoint's sum over a wave where the wave's pixels use many light lists: every lane at one entry, a few
distinct entries, the last count that the wave sums entry by entry, one past it, and every lane at an entry of its own;
lists inside the stage (256 entries) and beyond it (1024). References are the caller's, not the chain's.

Tolerance: relative L2 of 1e-3 against the FP64 adjoint per parameter group, the adjoint's documented bound.
"""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu

W, H, L, KEY_CAP, INDEX_CAP = 70, 45, 96, 64, 1024


@pytest.mark.parametrize("per_list", [4, 16])
@pytest.mark.parametrize("groups", [1, 2, 8, 9, 64])
def test_adjoint_of_waves_with_many_lists(oracle, vctx, groups, per_list):
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(W, H), ol.cfg(attenuation=1)
    pos, lig = co.synth_lights(77, L)
    lig[:, 3] = 60.0  # every light reaches most pixels
    depth, normals = co.synth_frame(4042, W, H, cam)
    ar, me = co.synth_materials(4042, W * H)
    rng = np.random.default_rng(groups)
    x, y = np.meshgrid(np.arange(W), np.arange(H))
    refs = ((x % 32 + 32 * (y % 2)) % groups).astype(np.uint32).reshape(-1)  # a wave covers two rows of 32 pixels
    counts = np.full(KEY_CAP, per_list, np.uint32)
    offsets = (np.arange(KEY_CAP) * per_list).astype(np.uint32)
    idx = np.concatenate([np.sort(rng.choice(L, per_list, replace=False)) for _ in range(KEY_CAP)]).astype(np.uint32)
    gout = rng.normal(0.0, 1.0, (W * H, 4)).astype(np.float32)
    g_pos, g_lig, g_ar = (to_dev(np.zeros((n, 4), np.float32)) for n in (L, L, W * H))
    vctx.shade_backward(W, H, cam, cf, to_dev(depth), to_dev(normals), to_dev(ar), to_dev(me), to_dev(refs), KEY_CAP,
                        to_dev(counts), to_dev(offsets), to_dev(idx), INDEX_CAP, to_dev(pos), to_dev(lig), L,
                        to_dev(gout), g_pos, g_lig, g_ar)
    want = co.shade_backward(W, H, cam, cf, depth, normals, ar, me, refs, KEY_CAP, counts, offsets, idx,
                             pos.astype(np.float64), lig.astype(np.float64), gout)
    got = [from_dev(g, np.float32, (n, 4)) for g, n in ((g_pos, L), (g_lig, L), (g_ar, W * H))]
    for a, b, cols in ((got[0], want[0], slice(0, 3)), (got[1], want[1], slice(0, 3)), (got[1], want[1], slice(3, 4)),
                       (got[2], want[2], slice(0, 3)), (got[2], want[2], slice(3, 4))):
        norm = np.linalg.norm(b[:, cols])
        assert norm > 0.0
        assert np.linalg.norm(a[:, cols] - b[:, cols]) <= 1e-3 * norm
