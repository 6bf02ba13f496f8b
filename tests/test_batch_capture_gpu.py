"""A batched run recorded into the caller's own graph. A run that could not be launched whole leaves the batch's work memory
to be cleared by the next one that runs, and a recorded one does not run: so what is recorded does not depend on it, and
replays and eager runs in any order give the bytes of the per-frame path."""
import ctypes

import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

W, H, L, F = 200, 120, 300, 3


def _batch(vctx):
    import torch
    import vren_amd
    cam = ol.camera(W, H)
    out = torch.zeros(F, W * H * 4, device="cuda")
    keep, descs = [out], []
    for f in range(F):
        t = {"depth": torch.empty(W * H, device="cuda"), "normals": torch.empty(W * H * 4, dtype=torch.int16, device="cuda"),
             "ar": torch.empty(W * H, 4, device="cuda"), "metal": torch.empty(W * H, device="cuda"),
             "pos": torch.empty(L, 4, device="cuda"), "lig": torch.empty(L, 4, device="cuda")}
        vctx.synth_frame(70 + f, W, H, cam, 64, t["depth"], t["normals"])
        vctx.synth_materials(80 + f, W * H, t["ar"], t["metal"])
        vctx.synth_lights(90 + f, L, t["pos"], t["lig"])
        d = vren_amd.FrameDesc()
        d.width, d.height, d.camera = W, H, cam
        d.depth, d.normals = t["depth"].data_ptr(), t["normals"].data_ptr()
        d.albedo_roughness, d.metallic = t["ar"].data_ptr(), t["metal"].data_ptr()
        d.light_positions, d.point_lights, d.light_count = t["pos"].data_ptr(), t["lig"].data_ptr(), L
        d.output = out[f].data_ptr()
        keep.append(t)
        descs.append(d)
    torch.cuda.synchronize()
    return vren_amd.Batch(vctx, descs, ol.cfg()), out, keep


def _ok(rc):
    assert rc == 0, rc


def _record(hip, batch, stream):
    """The graph of one batched run and its number of nodes."""
    graph, n = ctypes.c_void_p(), ctypes.c_size_t()
    _ok(hip.hipStreamBeginCapture(stream, 2))
    assert batch.ctx.lib.vren_batch_run(batch.h, stream, batch.BATCHED) == 0
    _ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
    _ok(hip.hipGraphGetNodes(graph, None, ctypes.byref(n)))
    return graph, n.value


def test_recorded_runs(vctx):
    import torch
    hip = ctypes.CDLL("libamdhip64.so")
    batch, out, keep = _batch(vctx)
    batch.run(batch.PER_FRAME)
    torch.cuda.synchronize()
    want = out.clone()
    stream = ctypes.c_void_p()
    _ok(hip.hipStreamCreate(ctypes.byref(stream)))
    # a run that cannot be launched: its capture is no longer valid
    _ok(hip.hipStreamBeginCapture(stream, 2))
    assert hip.hipStreamSynchronize(stream) != 0
    assert batch.ctx.lib.vren_batch_run(batch.h, stream, batch.BATCHED) != 0
    broken = ctypes.c_void_p()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(broken)) != 0
    hip.hipGetLastError()
    first, n = _record(hip, batch, stream)
    second, m = _record(hip, batch, stream)
    assert n == m
    execs = []
    for g in (first, second):
        e = ctypes.c_void_p()
        _ok(hip.hipGraphInstantiate(ctypes.byref(e), g, None, None, ctypes.c_size_t(0)))
        execs.append(e)

    def eager(mode):
        batch.run(mode)
        torch.cuda.synchronize()

    def replay(e):
        _ok(hip.hipGraphLaunch(e, stream))
        _ok(hip.hipStreamSynchronize(stream))

    for k, run in enumerate([lambda: eager(batch.BATCHED), lambda: replay(execs[0]), lambda: replay(execs[0]),
                             lambda: eager(batch.PER_FRAME), lambda: replay(execs[1]), lambda: eager(batch.GRAPH),
                             lambda: replay(execs[0]), lambda: eager(batch.GRAPH)]):
        out.zero_()
        torch.cuda.synchronize()
        run()
        assert np.array_equal(out.cpu().numpy(), want.cpu().numpy()), k
    for e in execs:
        _ok(hip.hipGraphExecDestroy(e))
    for g in (first, second):
        _ok(hip.hipGraphDestroy(g))
    _ok(hip.hipStreamDestroy(stream))
    batch.close()
