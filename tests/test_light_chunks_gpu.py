"""The light stage at the edges of its 4096-light chunks: codes, order and every BVH node bit for bit against the oracle,
for lights in random order, lights whose indices follow their places (a chunk's run lies inside one workgroup's range of
another run's codes) and lights all in one place (every code equal); and a batch that mixes frames of no light, one
chunk and several."""
import ctypes

import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu


def _lights(co, L, order):
    pos, lig = co.synth_lights(4242, max(L, 1))
    pos, lig = pos[:L], lig[:L]
    if order == "ordered":
        pos = pos[np.argsort(pos[:, 0], kind="stable")]
    elif order == "equal":
        pos = np.repeat(pos[:1], L, axis=0)
    return np.ascontiguousarray(pos), np.ascontiguousarray(lig)


def _same_nodes(got, want):
    return np.array_equal(got.view(np.uint32).reshape(-1, 8)[:, :7], want.view(np.uint32).reshape(-1, 8)[:, :7])


@pytest.mark.parametrize("order", ["random", "ordered", "equal"])
@pytest.mark.parametrize("L,bits", [(32, 5), (1024, 10), (1025, 5), (2049, 10), (4095, 5), (4096, 10), (4097, 10), (8192, 5),
                                    (8193, 10), (20000, 5), (70001, 10)])
def test_light_chunks(oracle, vctx, L, bits, order):
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(640, 360), ol.cfg(morton_bits=bits)
    pos, lig = _lights(co, L, order)
    nb = oracle.calc("buffer_length", L)
    vp, codes, bvh = empty_dev(16 * L), empty_dev(8 * L), empty_dev(32 * nb, fill=0xCD)
    vctx.construct_point_light_bvh(to_dev(pos), to_dev(lig), L, cam, cf, vp, codes, bvh)
    ovp, ocodes, obvh = co.light_bvh(pos, lig, cam, cf)
    assert np.array_equal(from_dev(vp, np.uint32, (L, 4)), ovp.view(np.uint32))
    assert np.array_equal(from_dev(codes, np.uint32, (L, 2)), ocodes)
    assert _same_nodes(from_dev(bvh, ol.BVH_DTYPE, (nb,)), obvh)


def test_batch_of_mixed_light_chunks(oracle, vctx):
    import torch
    import vren_amd
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(64, 64), ol.cfg()
    counts = [0, 300, 4096, 4097, 0, 1, 9000, 0]
    depth, normals = co.synth_frame(5, 64, 64, cam)
    ar, me = co.synth_materials(5, 64 * 64)
    shared = [to_dev(x) for x in (depth, normals, ar, me)]
    keep, descs = [shared], []
    for L in counts:
        pos, lig = _lights(co, L, "random")
        dev = (to_dev(pos) if L else None, to_dev(lig) if L else None, torch.zeros(64 * 64 * 4, device="cuda"))
        d = vren_amd.FrameDesc()
        d.width, d.height, d.camera = 64, 64, cam
        d.depth, d.normals, d.albedo_roughness, d.metallic = (x.data_ptr() for x in shared)
        if L:
            d.light_positions, d.point_lights = dev[0].data_ptr(), dev[1].data_ptr()
        d.light_count, d.output, d.key_capacity, d.index_capacity = L, dev[2].data_ptr(), 4096, 1 << 20
        keep.append(dev)
        descs.append(d)
    batch = vren_amd.Batch(vctx, descs, cf)
    for mode in (batch.BATCHED, batch.PER_FRAME, batch.GRAPH, batch.GRAPH):
        batch.run(mode)
        torch.cuda.synchronize()
        for f, L in enumerate(counts):
            if L == 0:
                continue
            pos, lig = _lights(co, L, "random")
            _, ocodes, obvh = co.light_bvh(pos, lig, cam, cf)
            o = batch.outputs(f)
            assert np.array_equal(_read(o.light_codes, 8 * L).view(np.uint32).reshape(L, 2), ocodes), (mode, L)
            assert _same_nodes(_read(o.bvh, 32 * o.bvh_length), obvh), (mode, L)
    batch.close()


def _read(ptr, nbytes):
    hip = ctypes.CDLL("libamdhip64.so")
    out = np.zeros(nbytes, np.uint8)
    assert hip.hipMemcpy(ctypes.c_void_p(out.ctypes.data), ctypes.c_void_p(ptr), ctypes.c_size_t(nbytes), ctypes.c_int(2)) == 0
    return out
