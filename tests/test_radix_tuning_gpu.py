"""Tuned choices of the radix sort for a few thousand keys: a table that names a configuration is followed there as for
more keys (seen from the launches of a recorded call), the tuner offers and stores the one-workgroup sort that an untuned
call takes, and that configuration sorts any number of keys."""
import ctypes

import numpy as np
import pytest

from gpu_util import empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu

ONE_WORKGROUP = 2  # the algorithm


def _launches(ctx, n):
    """The number of launches of one sort of n pairs."""
    hip = ctypes.CDLL("libamdhip64.so")
    keys, vals = empty_dev(4 * n, fill=7), empty_dev(4 * n)
    scratch = empty_dev(ctx.radix_sort_scratch_bytes(n, True))
    stream, graph, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    st = ctx.lib.vren_radix_sort(ctx.h, stream, *(ctypes.c_void_p(t.data_ptr()) for t in (keys, vals)), n, 0, 32,
                                 ctypes.c_void_p(scratch.data_ptr()), scratch.numel())
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0 and st == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    return nodes.value


def _sorted(ctx, n, values=True):
    keys = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    dk, dv = to_dev(keys), to_dev(np.arange(n, dtype=np.uint32)) if values else None
    ctx.radix_sort(dk, dv, n, empty_dev(ctx.radix_sort_scratch_bytes(n, values)))
    order = np.argsort(keys, kind="stable")
    return np.array_equal(from_dev(dk, np.uint32, (n,)), keys[order]) and (
        not values or np.array_equal(from_dev(dv, np.uint32, (n,)), order.astype(np.uint32)))


@pytest.mark.parametrize("n", [3000, 8192])
def test_a_tuned_choice_is_followed(tmp_path, n):
    import vren_amd
    ctx = vren_amd.Context(0)
    untuned = _launches(ctx, n)
    table = tmp_path / "tuned.txt"
    table.write_text("radix %d 8 23 16 0\n" % ((n.bit_length() - 1) << 8 | 1 << 7 | 32))
    ctx.check(ctx.lib.vren_autotune_load(ctx.h, str(table).encode()))
    assert untuned == 1 and _launches(ctx, n) >= 5  # a histogram and four passes
    assert _sorted(ctx, n)
    ctx.close()


def test_the_tuner_offers_what_an_untuned_call_takes(tmp_path):
    import vren_amd
    ctx = vren_amd.Context(0)
    best, ms = ctx.autotune_radix_sort(4096, True)
    assert ctx.radix_configs()[best][3] == ONE_WORKGROUP and ms > 0
    assert _launches(ctx, 4096) == 1 and _sorted(ctx, 4096)
    table = tmp_path / "tuned.txt"
    ctx.check(ctx.lib.vren_autotune_save(ctx.h, str(table).encode()))
    other = vren_amd.Context(0)
    other.check(other.lib.vren_autotune_load(other.h, str(table).encode()))
    assert _launches(other, 4096) == 1 and _sorted(other, 4096)
    best, _ = ctx.autotune_radix_sort(8193, True)  # another algorithm: its own launches are not timed a second time
    assert ctx.radix_configs()[best][3] != ONE_WORKGROUP
    other.close()
    ctx.close()


@pytest.mark.parametrize("n", [1, 2049, 8192, 8193, 100003, (1 << 19) + 1])
def test_the_one_workgroup_configuration_sorts_any_number(n):
    import vren_amd
    ctx = vren_amd.Context(0)
    ctx.radix_force_config([c[3] for c in ctx.radix_configs()].index(ONE_WORKGROUP))
    assert _sorted(ctx, n) and _sorted(ctx, n, values=False)
    ctx.close()
