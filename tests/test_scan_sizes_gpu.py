"""The exclusive scan around the length of one tile (16384 elements), below which a segment is scanned by one workgroup
without statuses: one and several segments, in place, from buffers off a 16-byte boundary; equal to the oracle."""
import ctypes

import numpy as np
import pytest

from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("blocks", [1, 5])
@pytest.mark.parametrize("n", [1, 3, 16383, 16384, 16385])
def test_scan_of_one_tile_segments(vctx, oracle, n, blocks, noalloc):
    x = np.random.default_rng(n).integers(0, 1 << 32, n * blocks, dtype=np.uint64).astype(np.uint32)
    want = np.concatenate([oracle.exclusive_scan_u32(x[b * n:(b + 1) * n]) for b in range(blocks)])

    def scan(a, b, n, blocks):
        if not noalloc:
            return vctx.exclusive_scan_u32(a, b, n, blocks)
        vctx.check(vctx.lib.vren_exclusive_scan_u32_noalloc(vctx.h, vctx.stream(), ctypes.c_void_p(a.data_ptr()),
                                                            ctypes.c_void_p(b.data_ptr()), n, blocks))

    for shift in (0, 1):
        src = to_dev(np.concatenate([np.zeros(shift, np.uint32), x]))[4 * shift:]
        out = empty_dev(4 * (x.size + shift))[4 * shift:]
        scan(src, out, n, blocks)
        assert np.array_equal(from_dev(out, np.uint32), want)
        scan(src, src, n, blocks)
        assert np.array_equal(from_dev(src, np.uint32), want)
