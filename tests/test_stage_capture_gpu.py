"""The stage calls captured into a graph on a context that has not assigned lights before, replayed around the program's own
eager assign_lights of a larger key capacity: the eager calls leave the memory of the captured ones where it was, and every
replay gives the oracle's clusters and lists."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

W, H, L = 333, 200, 700
KEY_CAP, INDEX_CAP = 1 << 14, 1 << 20


def _buffers(nb):
    return {"vp": empty_dev(16 * L), "codes": empty_dev(8 * L), "bvh": empty_dev(32 * nb), "keys": empty_dev(4 << 17),
            "count": empty_dev(4), "refs": empty_dev(4 * W * H), "counts": empty_dev(4 << 17), "offsets": empty_dev(4 << 17),
            "indices": empty_dev(4 * INDEX_CAP), "total": empty_dev(4)}


def _stages(ctx, cam, cf, g, b, key_cap):
    ctx.construct_point_light_bvh(g["pos"], g["lig"], L, cam, cf, b["vp"], b["codes"], b["bvh"])
    ctx.find_unique_cluster_list(W, H, cam, cf, g["depth"], g["normals"], b["keys"], key_cap, b["count"], b["refs"])


def _assign(ctx, cam, cf, b, key_cap):
    ctx.assign_lights(W, H, cam, cf, b["keys"], b["count"], key_cap, b["bvh"], L, b["codes"], b["vp"], b["counts"],
                      b["offsets"], b["indices"], INDEX_CAP, b["total"])


def test_captured_stage_calls_beside_eager_ones(oracle):
    import torch
    import vren_amd
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(W, H), ol.cfg()
    pos, lig = co.synth_lights(11, L)
    lig[:, 3] *= np.float32(3.0)
    nb = oracle.calc("buffer_length", L)
    ovp, ocodes, obvh = co.light_bvh(pos, lig, cam, cf)
    ctx = vren_amd.Context(0)
    g = {"pos": to_dev(pos), "lig": to_dev(lig)}
    frames = []
    for seed in (3, 4):
        depth, normals = co.synth_frame(seed, W, H, cam)
        okeys, n, orefs = co.unique_clusters(W, H, cam, cf, depth, normals)
        frames.append((to_dev(depth), to_dev(normals), okeys[:n], n, orefs) + co.assign(W, H, cam, cf, okeys, n, obvh, ocodes, ovp))
    g["depth"], g["normals"] = frames[0][0].clone(), frames[0][1].clone()
    b, eager = _buffers(nb), _buffers(nb)
    _stages(ctx, cam, cf, g, b, KEY_CAP)  # the scratch at its first size; no lights assigned yet
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _stages(ctx, cam, cf, g, b, KEY_CAP)
        _assign(ctx, cam, cf, b, KEY_CAP)
    spare = []
    for turn in range(4):
        depth, normals, okeys, n, orefs, oc, oo, oi, total = frames[turn % 2]
        g["depth"].copy_(depth)
        g["normals"].copy_(normals)
        graph.replay()
        torch.cuda.synchronize()
        assert int(from_dev(b["count"], np.uint32)[0]) == n and int(from_dev(b["total"], np.uint32)[0]) == total
        assert np.array_equal(from_dev(b["keys"], np.uint32, (n,)), okeys)
        assert np.array_equal(from_dev(b["refs"], np.uint32, (W * H,)), np.asarray(orefs).reshape(-1))
        assert np.array_equal(from_dev(b["counts"], np.uint32, (n,)), oc[:n])
        assert np.array_equal(from_dev(b["offsets"], np.uint32, (n,)), oo[:n])
        assert np.array_equal(from_dev(b["indices"], np.uint32, (total,)), oi[:total])
        # the program's own calls: every cluster of another frame with a slot, and memory that a freed block would become
        _stages(ctx, cam, cf, g, eager, 1 << 17)
        _assign(ctx, cam, cf, eager, 1 << 17)
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(eager["indices"], np.uint32, (total,)), oi[:total])
        spare.append(torch.full((1 << 20,), 0x5A, dtype=torch.uint8, device="cuda"))
    ctx.close()
