"""Morton codes of lights far outside a given box, and of boxes with degenerate axes: the light stage's quotient against the
division, on the CPU over dividends next to every cell border and extents of every magnitude, and the codes themselves
bit for bit against the oracle on the GPU."""
import ctypes

import numpy as np
import pytest

import oracle_lib as ol


def mismatches(oracle, r, ext, bits, planted=0):
    fn = oracle.lib.o_unit_quotient_mismatches
    fn.restype = ctypes.c_uint32
    r, ext = (np.ascontiguousarray(x, np.float32) for x in np.broadcast_arrays(r, ext))
    fused = ctypes.c_uint64()
    bad = fn(r.ctypes.data_as(ctypes.c_void_p), ext.ctypes.data_as(ctypes.c_void_p), ctypes.c_uint64(r.size),
             ctypes.c_uint32(bits), ctypes.c_uint32(planted), ctypes.byref(fused))
    return bad, fused.value


def near(x):
    """x and its neighbours in float."""
    x = np.asarray(x, np.float32)
    return np.concatenate([x, np.nextafter(x, np.float32(np.inf)), np.nextafter(x, np.float32(-np.inf))])


@pytest.mark.parametrize("bits", [1, 5, 10])
def test_quotient_in_the_cells_of_the_division(oracle, bits):
    rng = np.random.default_rng(bits)
    for e in (-149, -127, -61, -60, -59, -1, 0, 1, 59, 99, 100, 127):
        ext = np.ldexp(rng.uniform(1.0, 2.0, 200), e).astype(np.float32)
        cells = near(np.concatenate([np.arange(0, 1025) / 1024.0, rng.uniform(0, 1, 100)]))
        r = near((ext[:, None].astype(np.float64) * cells[None, :]).astype(np.float32).reshape(-1))
        x = np.tile(np.repeat(ext, cells.size), 3)
        bad, fused = mismatches(oracle, np.concatenate([r, -r]), np.concatenate([x, x]), bits)
        assert bad == 0, e
        assert (fused > 0) == (-60 <= e <= 99), (e, fused)


@pytest.mark.parametrize("bits", [5, 10])
def test_quotient_outside_the_box(oracle, bits):
    """Dividends far above the extent saturate as the division does: an overflow of the product is no NaN."""
    with np.errstate(over="ignore"):
        r = np.array([0.0, 1.0, -1.0, 4e8, -4e8, 1e20, -1e20, 3e38, np.inf, -np.inf, np.nan], np.float32)
        ext = np.array([0.0, -0.0, 1e-45, 1e-30, 1e-19, 1e-10, 1.0, -1.0, 1e10, 1e30, 3e38, np.inf, np.nan], np.float32)
        bad, _ = mismatches(oracle, r[:, None], ext[None, :], bits)
    assert bad == 0


def test_a_wrong_reciprocal_is_reported(oracle):
    ext = np.full(1025, 3.0, np.float32)
    assert mismatches(oracle, ext * (np.arange(1025, dtype=np.float32) / 1024), ext, 10, planted=1)[0] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("L,bits", [(1, 5), (100, 10), (4096, 5), (5000, 10)])
@pytest.mark.parametrize("lo,hi", [((0.0, 0.0, 0.0), (1e-30, 1e-19, 1.0)), ((-20.0, 0.0, 30.0), (20.0, 1e-38, 70.0)),
                                   ((-50.0, -50.0, 0.0), (50.0, 50.0, 100.0)), ((5.0, 5.0, 5.0), (5.0, 2.0, 1e30)),
                                   ((-1e30, 0.0, -1.0), (1e30, 1e35, 1.0))])
def test_codes_of_a_given_box(oracle, vctx, lo, hi, L, bits):
    from gpu_util import empty_dev, from_dev, to_dev
    co = ol.ClusteredOracle(oracle)
    cam = ol.camera(640, 360)
    cf = ol.cfg(morton_bits=bits, morton_aabb_mode=1, aabb=(lo, hi))
    pos, lig = co.synth_lights(77, L)
    pos = pos.copy()
    pos[::7, 0] *= np.float32(4e8)
    pos[::11, 1] *= np.float32(-1e20)
    nb = oracle.calc("buffer_length", L)
    vp, codes, bvh = empty_dev(16 * L), empty_dev(8 * L), empty_dev(32 * nb)
    vctx.construct_point_light_bvh(to_dev(pos), to_dev(lig), L, cam, cf, vp, codes, bvh)
    ovp, ocodes, _ = co.light_bvh(pos, lig, cam, cf)
    assert np.array_equal(from_dev(vp, np.uint32, (L, 4)), ovp.view(np.uint32))
    assert np.array_equal(from_dev(codes, np.uint32, (L, 2)), ocodes)
