"""assign_lights on made-up cluster keys, at the edges of the list writing: one cluster, a run of 256 clusters and one past
it, more clusters than one run of every workgroup holds, more than have list slots (their lists are traversed again),
lists longer than a slot, and an index buffer that ends inside the lists."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

W, H = 640, 360


@pytest.mark.parametrize("n,L,radius,room", [
    (1, 40, None, None), (255, 300, None, None), (256, 300, None, 100), (257, 300, 30.0, None), (3000, 600, 60.0, 70001),
    (33000, 64, None, None), (140000, 33, None, 5000)])
def test_assign_lists(oracle, vctx, n, L, radius, room):
    import vren_amd
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(W, H), ol.cfg()
    pos, lig = co.synth_lights(99, L)
    if radius:
        lig[:, 3] = radius
    vp, codes, bvh = co.light_bvh(pos, lig, cam, cf)
    rng = np.random.default_rng(n)
    keys = (rng.integers(0, 20, n) | (rng.integers(0, 12, n) << 8) | (rng.integers(0, 45, n) << 16) |
            (rng.integers(0, 54, n) << 26)).astype(np.uint32)
    oc, oo, oi, total = co.assign(W, H, cam, cf, keys, n, bvh, codes, vp)
    cap = room or max(total, 1)
    counts, offsets, tot = empty_dev(4 * n, fill=0xA5), empty_dev(4 * n, fill=0xA5), empty_dev(4)
    idx = empty_dev(4 * cap + 4, fill=0xA5)
    vctx.assign_lights(W, H, cam, cf, to_dev(keys), to_dev(np.array([n], np.uint32)), n, to_dev(bvh), L, to_dev(codes),
                       to_dev(vp), counts, offsets, idx, cap, tot)
    assert int(from_dev(tot, np.uint32)[0]) == total
    assert np.array_equal(from_dev(counts, np.uint32, (n,)), oc[:n])
    assert np.array_equal(from_dev(offsets, np.uint32, (n,)), oo[:n])
    got, m = from_dev(idx, np.uint32), min(total, cap)
    assert np.array_equal(got[:m], oi[:m]) and got[cap] == 0xA5A5A5A5
    if total > cap:
        with pytest.raises(vren_amd.VrenError):
            vctx.sync_status()
    else:
        vctx.sync_status()
