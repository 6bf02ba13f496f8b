"""Per-stage times of a batched run: a time for every stage that launches something in a normal run, and none for the others,
for tables with one launch for lights and clusters, with two, with frames of several light chunks and without lights."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

INIT, LIGHTS, LEAVES, UPPER, CLUSTERS, COUNTS, OFFSETS, LISTS, SHADE = range(9)


@pytest.mark.parametrize("W,H,L,stages", [
    (320, 180, 300, (LIGHTS, COUNTS, LISTS, SHADE)),
    (320, 180, 4100, (LIGHTS, LEAVES, UPPER, COUNTS, LISTS, SHADE)),
    (2560, 1440, 300, (LIGHTS, CLUSTERS, COUNTS, LISTS, SHADE)),
    (2560, 1440, 4100, (LIGHTS, LEAVES, UPPER, CLUSTERS, COUNTS, LISTS, SHADE)),
    (320, 180, 0, (CLUSTERS, COUNTS, SHADE))])
@pytest.mark.parametrize("concurrent", [0, 1])
def test_stages_of_a_run(vctx, W, H, L, stages, concurrent):
    import torch
    import vren_amd
    cam = ol.camera(W, H)
    t = {"depth": torch.empty(W * H, device="cuda"), "normals": torch.empty(W * H * 4, dtype=torch.int16, device="cuda"),
         "ar": torch.empty(W * H, 4, device="cuda"), "metal": torch.empty(W * H, device="cuda"),
         "pos": torch.empty(max(L, 1), 4, device="cuda"), "lig": torch.empty(max(L, 1), 4, device="cuda"),
         "out": torch.zeros(W * H, 4, device="cuda")}
    vctx.synth_frame(1, W, H, cam, 64, t["depth"], t["normals"])
    vctx.synth_materials(2, W * H, t["ar"], t["metal"])
    d = vren_amd.FrameDesc()
    d.width, d.height, d.camera, d.output = W, H, cam, t["out"].data_ptr()
    d.depth, d.normals = t["depth"].data_ptr(), t["normals"].data_ptr()
    d.albedo_roughness, d.metallic = t["ar"].data_ptr(), t["metal"].data_ptr()
    if L:
        vctx.synth_lights(3, L, t["pos"], t["lig"])
        d.light_positions, d.point_lights, d.light_count = t["pos"].data_ptr(), t["lig"].data_ptr(), L
    torch.cuda.synchronize()
    batch = vren_amd.Batch(vctx, [d], ol.cfg())
    if concurrent and L:  # lights on the second stream: a launch of their own, timed ahead of the clusters'
        batch.set_shape(1, 32, 8, 1)
        stages = sorted({*stages, CLUSTERS})
    for _ in range(2):
        t["out"].zero_()
        ms = batch.run_profiled()
        assert [i for i in range(9) if ms[i] > 0] == list(stages), ms
        image = t["out"].clone()
        t["out"].zero_()
        batch.run(batch.BATCHED)
        torch.cuda.synchronize()
        assert np.array_equal(t["out"].cpu().numpy(), image.cpu().numpy())
    batch.close()
