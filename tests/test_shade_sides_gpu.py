"""The side test that the forward shade and its adjoint take before a light's distance: lights in front of, behind and
in a pixel's plane, at the pixel itself, just inside and just outside their radius, and directional lights that are not
of unit length; lists inside the stage (256 entries) and past it, both attenuations.

Tolerances: 1e-5 relative (floor 1e-6) against the FP64 oracle for the radiance, a relative L2 of 1e-3 per
parameter group for the adjoint: the documented bounds of the two.
"""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

W, H, KEY_CAP = 45, 27, 1


def flat_frame(co):
    """A wall at z = 0 facing the camera at z = -50: world position (x, y, 0) of each pixel, and the buffers."""
    cam, near, far = ol.camera(W, H), 0.1, 100.0
    depth = np.full(W * H, (far / (far - near)) * (1.0 - near / 50.0), np.float32)
    z = -(far * near) / (far - near) / (float(depth[0]) - far / (far - near))
    x, y = np.meshgrid(np.arange(W), np.arange(H))
    px = ((x / W * 2 - 1) * W / H * z).reshape(-1)
    py = (((1 - y / H) * 2 - 1) * z).reshape(-1)
    normals = np.tile(np.array([0.0, 0.0, -1.0, 0.0], np.float16), (W * H, 1)).view(np.uint16)
    return cam, depth, np.ascontiguousarray(normals), np.stack([px, py, np.full(W * H, z - 50.0)], axis=1)


def lights_around(point, at_pixel):
    x, y, z = point
    rows = [(x + 0.3, y, z - 0.5, 4.0), (x, y + 0.4, z + 0.5, 4.0), (x + 1.0, y, z, 4.0), (x - 2.0, y, z - 1e-4, 4.0),
            (x, y, z - 1.999998, 2.0), (x, y, z - 2.000002, 2.0), (x + 0.2, y + 0.2, z + 1e-4, 4.0), (x, y, z - 1.0, 0.0)]
    if at_pixel:
        rows.append((x, y, z, 3.0))
    rows = np.array(rows, np.float32)
    pos, lig = np.zeros((len(rows), 4), np.float32), np.zeros((len(rows), 4), np.float32)
    pos[:, :3], lig[:, 3] = rows[:, :3], rows[:, 3]
    lig[:, :3] = np.random.default_rng(5).uniform(0.2, 1.0, (len(rows), 3))
    return pos, lig


def one_list(n, copies):
    idx = np.tile(np.arange(n, dtype=np.uint32), copies)
    return np.zeros(W * H, np.uint32), np.array([idx.size], np.uint32), np.zeros(1, np.uint32), idx


@pytest.mark.parametrize("copies", [1, 60])
@pytest.mark.parametrize("atten", [0, 1])
def test_forward_sides(oracle, vctx, atten, copies):
    co = ol.ClusteredOracle(oracle)
    cam, depth, normals, points = flat_frame(co)
    cf = ol.cfg(attenuation=atten)
    pos, lig = lights_around(points[(H // 2) * W + W // 2], True)
    refs, counts, offsets, idx = one_list(len(pos), copies)
    ar, me = co.synth_materials(9, W * H)
    dirs = np.zeros((4, 4), np.float32)
    dirs[0, :3], dirs[1, :3] = (0.3, -0.4, 2.5), (0.5, 0.6, 0.7)
    dirs[2, :3], dirs[3, :3] = (0.0, 0.1, -3.0), (0.9, 0.9, 0.9)
    out = empty_dev(16 * W * H, fill=0xFF)
    vctx.shade(W, H, cam, cf, to_dev(depth), to_dev(normals), to_dev(ar), to_dev(me), to_dev(refs), KEY_CAP,
               to_dev(counts), to_dev(offsets), to_dev(idx), idx.size, to_dev(pos), to_dev(lig), len(pos), out,
               to_dev(dirs), 2)
    got = from_dev(out, np.float32, (W * H, 4))
    want, mask = co.shade(W, H, cam, cf, depth, normals, ar, me, refs, KEY_CAP, counts, offsets, idx, pos, lig,
                          dirl=dirs.reshape(2, 8))
    assert mask.all()
    err = np.abs(got[:, :3] - want[:, :3]) / np.maximum(np.abs(want[:, :3]), 0.1)
    assert err.max() <= 1e-5, err.max()


@pytest.mark.parametrize("copies", [1, 70])
def test_adjoint_sides(oracle, vctx, copies):
    co = ol.ClusteredOracle(oracle)
    cam, depth, normals, points = flat_frame(co)
    cf = ol.cfg(attenuation=1)
    pos, lig = lights_around(points[(H // 2) * W + W // 2], False)
    L = len(pos)
    refs, counts, offsets, idx = one_list(L, copies)
    ar, me = co.synth_materials(9, W * H)
    gout = np.random.default_rng(3).normal(0.0, 1.0, (W * H, 4)).astype(np.float32)
    grads = [to_dev(np.zeros((n, 4), np.float32)) for n in (L, L, W * H)]
    vctx.shade_backward(W, H, cam, cf, to_dev(depth), to_dev(normals), to_dev(ar), to_dev(me), to_dev(refs), KEY_CAP,
                        to_dev(counts), to_dev(offsets), to_dev(idx), idx.size, to_dev(pos), to_dev(lig), L, to_dev(gout),
                        *grads)
    want = co.shade_backward(W, H, cam, cf, depth, normals, ar, me, refs, KEY_CAP, counts, offsets, idx,
                             pos.astype(np.float64), lig.astype(np.float64), gout)
    got = [from_dev(g, np.float32, (n, 4)) for g, n in zip(grads, (L, L, W * H))]
    for a, b, cols in ((got[0], want[0], slice(0, 3)), (got[1], want[1], slice(0, 3)), (got[1], want[1], slice(3, 4)),
                       (got[2], want[2], slice(0, 3)), (got[2], want[2], slice(3, 4))):
        norm = np.linalg.norm(b[:, cols])
        assert norm > 0.0 and np.linalg.norm(a[:, cols] - b[:, cols]) <= 1e-3 * norm
    behind = [1, 7]  # behind the wall by 0.5; radius 0
    assert not got[0][behind].any() and not got[1][behind].any()
