"""Cluster keys over cameras: which pixels take the short form of the depth slice is decided from a bound that depends on the
planes and on the slices per unit of ln z, so planes close together and far apart, near planes from 1e-30 to 1e3, narrow
and wide fields of view and the fewest and most slices are compared with the oracle bit for bit, over depths next to the
slices' borders and runs of consecutive floats."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev
from test_cluster_keys_gpu import border_depths

pytestmark = pytest.mark.gpu

KEY_CAP = 1 << 20
W, H = 417, 500


def depths(rng, n, near, far, steps):
    d = border_depths(rng, n, near, far, steps)
    starts = np.concatenate([rng.choice(d[np.isfinite(d)], 400), rng.random(400).astype(np.float32),
                             np.array([0.0, 1.0, np.nextafter(np.float32(1), np.float32(0))], np.float32)])
    runs = (starts.view(np.uint32)[:, None] + np.arange(-40, 41, dtype=np.int64)[None, :]).astype(np.uint32).reshape(-1)
    d[:runs.size] = runs.view(np.float32)
    return rng.permutation(d)


@pytest.mark.parametrize("fov", [4.0, 90.0, 170.0])
@pytest.mark.parametrize("slices", [None, 1, 255, 256])
@pytest.mark.parametrize("near,far", [(0.1, 100.0), (1e-3, 1e4), (1.0, 10.0), (1.0, 1.03), (50.0, 51.0), (1e3, 1e6), (1e-6, 1e6),
                                      (0.9, 1.1), (1e-30, 1e30), (3e-39, 1.0), (1.0, np.inf)])
def test_keys_of_cameras(oracle, vctx, near, far, slices, fov):
    co = ol.ClusteredOracle(oracle)
    cam, n = ol.camera(W, H, fov_deg=fov, near=near, far=far), W * H
    rng = np.random.default_rng(7)
    cf = ol.cfg(key_mode=1, depth_slices=slices) if slices else ol.cfg()
    with np.errstate(all="ignore"):
        steps = slices or 2.0 / np.tan(np.deg2rad(fov) / 2) * 16 * np.log(min(far, 1e30) / near)
        depth = depths(rng, n, near, min(far, 1e30), max(1.0, steps))
    normals = np.zeros((n, 4), np.float16)
    normals[:, 2] = 1.0
    normals = normals.view(np.uint16)
    keys, count, refs = empty_dev(4 * KEY_CAP), empty_dev(4), empty_dev(4 * n)
    vctx.find_unique_cluster_list(W, H, cam, cf, to_dev(depth), to_dev(normals), keys, KEY_CAP, count, refs)
    want_keys, want_count, want_refs = co.unique_clusters(W, H, cam, cf, depth, normals)
    assert int(from_dev(count, np.uint32)[0]) == want_count
    assert np.array_equal(from_dev(keys, np.uint32)[:want_count], want_keys)
    assert np.array_equal(from_dev(refs, np.uint32), want_refs)
