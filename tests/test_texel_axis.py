"""The short form of the texel selection (include/vren_hip/sampler.h: vren_texel_axis_near) against the general one: the same
texels and the same weight's bits for every filter, address mode and texture side, at texel centres and edges, at
multiples of the side and their neighbours in float, at random coordinates and at the ends of the short form's range, with
a reciprocal that is off by an ulp either way."""
import ctypes

import numpy as np
import pytest


def coordinates(size):
    rng = np.random.default_rng(size)
    edge = np.concatenate([np.arange(-9, 10), rng.integers(-(1 << 22), 1 << 22, 4000),
                           np.array([-(1 << 22), 1 << 22]), size * np.arange(-40, 41)])
    edge = np.unique(np.concatenate([edge, edge + 0.5, edge - 0.5])) / size
    s = np.concatenate([edge, rng.uniform(-3.0, 3.0, 4000), rng.uniform(-1.0, 1.0, 4000) * (1 << 22) / size]).astype(np.float32)
    s = np.concatenate([s, np.nextafter(s, np.float32(np.inf)), np.nextafter(s, np.float32(-np.inf)),
                        np.array([0.0, -0.0, 1e-30, -1e-30], np.float32)])
    return np.ascontiguousarray(s)


def mismatches(oracle, s, size, filt, mode, ulps, planted=0):
    fn = oracle.lib.o_texel_axis_mismatches
    fn.restype = ctypes.c_uint32
    return fn(s.ctypes.data_as(ctypes.c_void_p), ctypes.c_uint64(s.size), ctypes.c_uint32(size), ctypes.c_uint32(filt),
              ctypes.c_uint32(mode), ctypes.c_int32(ulps), ctypes.c_uint32(planted))


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("filt", [0, 1])
def test_short_form_picks_the_same_texels(oracle, filt, mode):
    for size in (1, 2, 3, 5, 7, 33, 64, 97, 128, 255, 256, 1000, 4096, 10007, (1 << 20) + 7, (1 << 22) - 1, 1 << 22):
        s = coordinates(size)
        for ulps in (-1, 0, 1):
            if ulps and size & (size - 1) == 0:
                continue  # the reciprocal of a power of two is exact
            assert mismatches(oracle, s, size, filt, mode, ulps) == 0, (size, ulps)


def test_a_wrong_reciprocal_is_reported(oracle):
    assert mismatches(oracle, coordinates(97), 97, 1, 0, 0, planted=1) > 0
