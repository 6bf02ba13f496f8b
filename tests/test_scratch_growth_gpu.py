"""A scan captured over a fresh context's scratch, replayed around eager calls that outgrow it: bucket sorts of a little more
than the first megabyte, of several and of more than the blocks that are kept. The graph is replayed while its block is
kept, each time on other keys."""
import numpy as np
import pytest

from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

N = 70_001  # several tiles: the scan takes tickets and look-back words from the scratch


def _bucket_sort(ctx, oracle, n):
    keys = oracle.pcg32(n, 3, n)
    pairs = np.stack([keys, np.arange(n, dtype=np.uint32)], axis=1)
    out, starts = empty_dev(8 * n), empty_dev(4 << 8)
    ctx.bucket_sort(to_dev(pairs), n, out, starts, 256, 0)
    got = from_dev(out, np.uint32, (n, 2))
    assert np.array_equal(got, pairs[np.argsort(keys & 255, kind="stable")])


def test_captured_scan_beside_calls_that_outgrow_its_scratch(oracle):
    import torch
    import vren_amd
    ctx = vren_amd.Context(0)
    assert ctx.radix_sort_scratch_bytes(113_000, True) > 1 << 20
    x, out = empty_dev(4 * N), empty_dev(4 * N)
    x.zero_()
    ctx.exclusive_scan_u32(x, out, N)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.exclusive_scan_u32(x, out, N)
    spare = []
    for turn, n in enumerate((113_000, 300_000, 2_000_000, 9_000_000)):
        _bucket_sort(ctx, oracle, n)
        spare.append(torch.full((1 << 21,), 0x5A, dtype=torch.uint8, device="cuda"))
        keys = oracle.pcg32(turn, 5, N)
        x.copy_(to_dev(keys))
        graph.replay()
        assert np.array_equal(from_dev(out, np.uint32, (N,)), oracle.exclusive_scan_u32(keys, 1)), n
    _bucket_sort(ctx, oracle, 20_000_000)  # past a block that is not kept
    ctx.close()
