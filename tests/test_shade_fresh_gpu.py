"""The differentiable shade into buffers whose contents do not matter: the same radiance as into zeros, bit for bit, also
on background pixels; the same material gradient bit for bit, and the light gradients up to the order of their atomic
sums (relative L2 of 1e-4; each is a sum of at most a few thousand float terms); and autograd over tensors with more
rows than the frame has pixels or lights.
"""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu


def frame(oracle, vctx, W, H, L):
    from test_clustered_gpu import run_assign
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(W, H), ol.cfg(attenuation=1)
    depth, normals = co.synth_frame(5, W, H, cam)
    depth = depth.reshape(H, W)
    depth[: H // 3, : W // 2] = 1.0  # background
    ar, me = co.synth_materials(5, W * H)
    pos, lig = co.synth_lights(6, max(L, 1))
    lig[:, 3] *= 3.0
    g = run_assign(vctx, co, W, H, cam, cf, depth.reshape(-1), normals, pos, lig)
    return cam, cf, to_dev(depth), to_dev(normals), to_dev(ar), to_dev(me), g["dev"], to_dev(pos), to_dev(lig)


@pytest.mark.parametrize("W,H,L", [(1, 1, 1), (33, 31, 0), (70, 45, 700), (257, 130, 64)])
def test_fresh_equals_cleared(oracle, vctx, W, H, L):
    cam, cf, depth, normals, ar, me, d, pos, lig = frame(oracle, vctx, W, H, L)
    n, lists = W * H, (d["refs"], 1 << 20, d["counts"], d["offsets"], d["idx"], 1 << 22)
    gout = to_dev(np.random.default_rng(1).normal(size=(n, 4)).astype(np.float32))
    res = []
    for fresh, fill in ((False, 0), (True, 0xFF)):
        out, g_ar = empty_dev(16 * n, fill), empty_dev(16 * n, fill)
        g_pos, g_lig = empty_dev(16 * max(L, 1), fill), empty_dev(16 * max(L, 1), fill)
        vctx.shade(W, H, cam, cf, depth, normals, ar, me, *lists, pos, lig, L, out, fresh=fresh)
        vctx.shade_backward(W, H, cam, cf, depth, normals, ar, me, *lists, pos, lig, L, gout, g_pos, g_lig, g_ar,
                            fresh=fresh)
        res.append([from_dev(x, np.float32) for x in (out, g_ar, g_pos[:16 * L], g_lig[:16 * L])])
    for a, b in zip(res[0][:2], res[1][:2]):
        assert np.array_equal(a, b)
    for a, b in zip(res[0][2:], res[1][2:]):
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(a)


def test_autograd_with_spare_rows(oracle, vctx):
    import torch
    from vren_amd.autograd import ShadeFrame, shade
    W, H, L = 70, 45, 50
    cam, cf, depth, normals, ar, me, d, pos, lig = frame(oracle, vctx, W, H, L)
    f = ShadeFrame(vctx, W, H, cam, cf, depth, normals, me, d["refs"], 1 << 20, d["counts"], d["offsets"], d["idx"], 1 << 22)
    rows = lambda t: t.view(torch.float32).reshape(-1, 4)  # noqa: E731
    grads = []
    for spare in (0, 3):
        pad = torch.ones(spare, 4, device="cuda")
        p = [torch.cat([rows(t), pad]).requires_grad_(True) for t in (ar, pos, lig)]
        image = shade(p[1][:L] if spare else p[1], p[2], p[0], f)
        grads.append(torch.autograd.grad(image.square().sum(), p))
    for a, b in zip(*grads):
        assert torch.isfinite(b).all() and not b[a.shape[0]:].any()
        assert torch.linalg.norm(a - b[:a.shape[0]]) <= 1e-4 * torch.linalg.norm(a)
