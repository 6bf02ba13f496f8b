"""The cluster stage's short forms of a pixel's slice and normal code and its loads of whole rows: screens whose rows start at
every alignment, below and above one workgroup per CU, buffers that start 4 bytes past a 16-byte boundary, zero
normals, infinities, NaNs, depths at the slices' borders, in front of the near plane and past the far one; keys, counts
and references bit for bit against the oracle.
"""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

KEY_CAP = 1 << 20


def border_depths(rng, n, near, far, steps):
    """Depths whose view depths are spread over the slices, half of them next to a border."""
    k = rng.uniform(-1.0, steps + 1.0, n)
    k = np.where(rng.random(n) < 0.5, np.round(k) + rng.uniform(-3e-5, 3e-5, n), k)
    z = near * np.exp(k * np.log(far / near) / steps)
    return (far / (far - near) * (1.0 - near / z)).astype(np.float32)


def odd_normals(rng, n):
    v = rng.normal(size=(n, 4))
    v[:, :3] /= np.linalg.norm(v[:, :3], axis=1, keepdims=True)
    h = v.astype(np.float16)
    pick = rng.random((n, 3))
    h[:, :3] = np.where(pick < 0.15, np.float16(0.0), h[:, :3])
    h[rng.random(n) < 0.2, :3] = 0.0
    h[rng.random(n) < 0.1, 0] = -0.0
    for value in (np.inf, -np.inf, np.nan, 6e-8, 65504.0):
        rows = rng.random(n) < 0.01
        h[rows, rng.integers(0, 3, rows.sum())] = value
    third = rng.random(n) < 0.05                                 # components in ratios of exactly a third
    h[third, :3] = np.array([0.75, 0.25, -0.25], np.float16)[rng.permuted(np.tile(np.arange(3), (third.sum(), 1)), axis=1)]
    return np.ascontiguousarray(h).view(np.uint16)


@pytest.mark.parametrize("mode", ["reference", "sliced"])
@pytest.mark.parametrize("W,H,shift", [(1, 1, 0), (31, 33, 1), (64, 64, 1), (129, 70, 0), (1366, 101, 0), (1026, 64, 1),
                                       (2051, 1090, 0), (2080, 1088, 1)])
def test_keys_of_ragged_screens(oracle, vctx, W, H, shift, mode):
    co = ol.ClusteredOracle(oracle)
    cam, n = ol.camera(W, H), W * H
    rng = np.random.default_rng(W)
    cf = ol.cfg(key_mode=1, depth_slices=57) if mode == "sliced" else ol.cfg()
    depth, normals = border_depths(rng, n, 0.1, 100.0, 57), odd_normals(rng, n)
    flat = rng.random(n) < 0.3
    depth[flat], normals[flat] = 1.0, 0                           # cleared background
    pad = lambda a: to_dev(np.concatenate([np.zeros(4 * shift, np.uint8), np.ascontiguousarray(a).view(np.uint8).reshape(-1)]))  # noqa: E731
    d, nn, refs = pad(depth), pad(normals), empty_dev(4 * (n + shift))
    keys, count = empty_dev(4 * KEY_CAP), empty_dev(4)
    at = lambda t: t[4 * shift:]                                  # noqa: E731
    vctx.find_unique_cluster_list(W, H, cam, cf, at(d), at(nn), keys, KEY_CAP, count, at(refs))
    want_keys, want_count, want_refs = co.unique_clusters(W, H, cam, cf, depth, normals)
    U = int(from_dev(count, np.uint32)[0])
    assert U == want_count
    assert np.array_equal(from_dev(keys, np.uint32)[:U], want_keys)
    assert np.array_equal(from_dev(refs, np.uint32)[shift:], want_refs)
