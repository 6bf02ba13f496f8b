"""Light lists of a batch whose runs are shared by a team of four or two workgroups, or taken by one: lists longer than a slot beside
short ones and frames without lights, bit for bit against the oracle, and the same image as from one frame at a time."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import to_dev
from test_light_chunks_gpu import _read

pytestmark = pytest.mark.gpu

W, H = 130, 97


@pytest.mark.parametrize("frames", [1, 2, 5, 9, 64, 520])
def test_long_lists_of_a_batch(oracle, vctx, frames):
    import torch
    import vren_amd
    co = ol.ClusteredOracle(oracle)
    cam, cf = ol.camera(W, H), ol.cfg()
    kinds = []
    for k, (L, scale) in enumerate([(1500, 12.0), (0, 1.0), (700, 1.0), (5000, 5.0)]):
        pos, lig = co.synth_lights(40 + k, max(L, 1))
        lig[:, 3] *= np.float32(scale)
        depth, normals = co.synth_frame(50 + k, W, H, cam)
        ar, me = co.synth_materials(60 + k, W * H)
        dev = [to_dev(x) for x in (depth, normals, ar, me, pos, lig)]
        want = None
        if L:
            vp, codes, bvh = co.light_bvh(pos, lig, cam, cf)
            keys, n, _ = co.unique_clusters(W, H, cam, cf, depth, normals)
            want = (n,) + co.assign(W, H, cam, cf, keys, n, bvh, codes, vp, index_cap=1 << 22)
            if scale > 1:
                assert want[1].max() > 192
        kinds.append((L, dev, want))
    out = torch.zeros(frames, W * H * 4, device="cuda")
    descs = []
    for f in range(frames):
        L, dev, want = kinds[f % 4]
        d = vren_amd.FrameDesc()
        d.width, d.height, d.camera = W, H, cam
        d.depth, d.normals, d.albedo_roughness, d.metallic = (x.data_ptr() for x in dev[:4])
        if L:
            d.light_positions, d.point_lights = dev[4].data_ptr(), dev[5].data_ptr()
        d.light_count, d.output, d.key_capacity, d.index_capacity = L, out[f].data_ptr(), 4096, 1 << 20
        descs.append(d)
    batch = vren_amd.Batch(vctx, descs, cf)
    batch.run(batch.BATCHED)
    torch.cuda.synchronize()
    image = out.clone()
    for f in sorted(set(list(range(min(frames, 8))) + [frames - 1])):
        L, _, want = kinds[f % 4]
        o = batch.outputs(f)
        if not L:
            continue
        n, oc, oo, oi, total = want
        assert total < 1 << 20
        assert int(_read(o.assigned_total, 4).view(np.uint32)[0]) == total
        assert np.array_equal(_read(o.light_counts, 4 * n).view(np.uint32), oc[:n]), f
        assert np.array_equal(_read(o.light_offsets, 4 * n).view(np.uint32), oo[:n]), f
        assert np.array_equal(_read(o.light_indices, 4 * total).view(np.uint32), oi[:total]), f
    out.zero_()
    batch.run(batch.PER_FRAME)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), image.cpu().numpy())
    batch.close()
