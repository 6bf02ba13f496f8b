"""The material resolve of waves that share one material (scalar records), of waves that cross from one to the next
and of waves with a material per pixel; material and texture indices past their tables; texcoords inside and outside the
range of the short texel selection, and not finite. Read back through the ambient term as the albedo.

Tolerance: 1e-5 relative with a floor of 1e-2, the documented bound of the resolve against the FP64 oracle.
"""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev
from test_next_gpu import DeviceMaterials, make_materials, synth_texcoords

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reach", ["near", "far"])
@pytest.mark.parametrize("layout", ["one", "columns", "rows", "random"])
def test_resolve_by_wave(oracle, vctx, layout, reach):
    import vren_amd
    co = ol.ClusteredOracle(oracle)
    W, H = 197, 101
    cam = ol.camera(W, H)
    depth, normals = np.full(W * H, 0.9985, np.float32), co.synth_frame(7, W, H, cam)[1]
    textures, mats = make_materials(21)
    mats[1].base_color_texture_idx = 99              # past the texture table: zeros
    mats[2].metallic_roughness_texture_idx = mats[2].base_color_texture_idx
    tc, random_mi = synth_texcoords(22, W, H, len(mats))
    y, x = np.divmod(np.arange(W * H), W)
    mi = {"one": np.full(W * H, 5), "columns": (x // 13) % 10, "rows": (y // 3) % 8, "random": random_mi}[layout].astype(np.uint16)
    if reach == "far":
        rng = np.random.default_rng(23)
        tc = (tc * rng.choice([1.0, 1e3, 2.0 ** 15, 2.0 ** 20, 1e9], (W * H, 1))).astype(np.float32)
        tc[::97, 0], tc[::101, 1], tc[::103, 0] = np.nan, np.inf, -np.inf
    dm = DeviceMaterials(vren_amd, tc, mi, textures, mats)
    out = empty_dev(16 * W * H, fill=0xFF)
    zero, refs = to_dev(np.zeros(4, np.uint32)), to_dev(np.zeros(W * H, np.uint32))
    vctx.shade_materials(W, H, cam, ol.cfg(), to_dev(depth), to_dev(normals), dm.set, refs, 1, zero, zero, zero, 1, None,
                         None, 0, out)
    got = from_dev(out, np.float32, (W * H, 4))
    want = co.resolve_materials(tc, mi, mats, textures)[0][:, :3]
    albedo = np.power(got[:, :3].astype(np.float64), 2.2) / 0.03
    err = np.abs(albedo - want) / np.maximum(want, 1e-2)
    # past 2^24 texels the float remainder may leave [0, side), and its conversion to an index is the platform's: an
    # index inside the texture, but not the oracle's
    u = np.where(np.isfinite(tc), np.abs(tc), 0.0) * np.array([max(t[0].shape[1 - k] for t in textures) for k in (0, 1)])
    assert np.isfinite(albedo).all()
    err = err[(u < 2.0 ** 24).all(axis=1)]
    assert err.size > W * H
    assert err.max() <= 1e-5, (layout, reach, int(err.max(axis=1).argmax()), err.max())
