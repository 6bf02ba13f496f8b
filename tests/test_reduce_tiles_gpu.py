"""The up-sweep tree where its tiles change: one row of 1024 threads (up to 4096 values, 1024 float4), tiles of 16384 values
(4096 float4), second passes of one row and of a whole tile, inputs that end inside a row or on none, and segments that
start on any 4-byte boundary; every padded element equal to the oracle's."""
import numpy as np
import pytest

import vren_amd
from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 1023, 4095, 4096, 4097, 8191, 16384, 16385, 20481, 65535, (1 << 20) + 3])
@pytest.mark.parametrize("op", [vren_amd.REDUCE_ADD, vren_amd.REDUCE_MIN, vren_amd.REDUCE_MAX])
@pytest.mark.parametrize("blocks", [1, 3])
def test_reduce_tree_tiles(vctx, oracle, n, op, blocks):
    x = np.random.default_rng(n + op).integers(0, 1 << 32, n * blocks, dtype=np.uint64).astype(np.uint32)
    p = 1 << (n - 1).bit_length() if n > 1 else 1
    for shift in (0, 1):
        src = to_dev(np.concatenate([np.zeros(shift, np.uint32), x]))[4 * shift:]
        out = empty_dev(4 * (p * blocks + shift), fill=0xA5)[4 * shift:]
        vctx.reduce_u32(src, n, out, op, blocks)
        got = from_dev(out, np.uint32, (blocks, p))
        for b in range(blocks):
            assert np.array_equal(got[b], oracle.reduce_tree_u32(x[b * n:(b + 1) * n], op))


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 4097, (1 << 22) + 5])
@pytest.mark.parametrize("op", [vren_amd.REDUCE_ADD, vren_amd.REDUCE_MIN, vren_amd.REDUCE_MAX])
def test_reduce_vec4_tiles(vctx, oracle, n, op):
    x = np.random.default_rng(n + op).standard_normal((n, 4)).astype(np.float32)
    p = 1 << (n - 1).bit_length() if n > 1 else 1
    out = empty_dev(16 * p, fill=0xA5)
    vctx.reduce_vec4(to_dev(x), n, out, op)
    assert np.array_equal(from_dev(out, np.uint32, (p, 4)), oracle.reduce_tree_vec4(x, op).view(np.uint32))
