"""The radix and bucket sorts at the sizes where their path changes -- one workgroup up to 8192 keys, histogram parts up to
2^19, and the default tile's steps (2^19, 2^21, 15360 * 256 on 256 CUs) -- bit for bit against the oracle's stable
sorts, with keys of few and of many distinct values."""
import numpy as np
import pytest

from gpu_util import empty_dev, from_dev, to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("values", [True, False])
@pytest.mark.parametrize("n,begin,end,distinct", [
    (1, 0, 32, 1 << 32), (64, 0, 32, 3), (65, 5, 13, 1 << 32), (1023, 0, 32, 1 << 32), (1025, 0, 30, 7),
    (2048, 31, 32, 1 << 32), (2049, 0, 15, 1 << 32), (8191, 0, 32, 1), (8192, 0, 32, 1 << 32), (8193, 0, 32, 1 << 32),
    (40001, 3, 19, 1 << 32), ((1 << 19) - 1, 0, 32, 1 << 32), (1 << 19, 0, 30, 50), ((1 << 19) + 1, 0, 32, 1 << 32),
    ((1 << 21) + 1, 0, 16, 1 << 32), (15360 * 256 + 1, 0, 8, 1 << 32)])
def test_radix_sort_path_edges(oracle, vctx, n, begin, end, distinct, values):
    rng = np.random.default_rng(n)
    pool = rng.integers(0, 1 << 32, min(distinct, n), dtype=np.uint64).astype(np.uint32)
    keys = pool[rng.integers(0, pool.size, n)] if distinct <= n else rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    vals = np.arange(n, dtype=np.uint32)[::-1].copy() if values else None
    dk, dv = to_dev(keys), to_dev(vals) if values else None
    scratch = empty_dev(vctx.radix_sort_scratch_bytes(n, values), fill=0xA5)
    vctx.radix_sort(dk, dv, n, scratch, begin, end)
    ok, ov = oracle.stable_sort_kv(keys, vals, begin, end)
    assert np.array_equal(from_dev(dk, np.uint32, (n,)), ok)
    if values:
        assert np.array_equal(from_dev(dv, np.uint32, (n,)), ov)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 1000, 2049, 8192, 8193, 65535, 65536, 70000, (1 << 19) + 1])
@pytest.mark.parametrize("buckets,shift,distinct", [(65536, 0, 1 << 32), (65536, 16, 5), (256, 28, 1 << 32), (2, 0, 1)])
def test_bucket_sort_path_edges(oracle, vctx, n, buckets, shift, distinct):
    rng = np.random.default_rng(n + shift)
    pool = rng.integers(0, 1 << 32, min(distinct, n), dtype=np.uint64).astype(np.uint32)
    pairs = np.stack([pool[rng.integers(0, pool.size, n)], np.arange(n, dtype=np.uint32)], axis=1)
    out, starts = empty_dev(8 * n), empty_dev(4 * buckets, fill=0xA5)
    vctx.bucket_sort(to_dev(pairs), n, out, starts, buckets, shift)
    opairs, ostarts = oracle.bucket_sort(pairs, buckets, shift)
    assert np.array_equal(from_dev(out, np.uint32, (n, 2)), opairs)
    assert np.array_equal(from_dev(starts, np.uint32, (buckets,)), ostarts)


def test_scratch_for_more_keys_is_enough_for_fewer():
    import vren_amd
    lib = vren_amd.lib()
    for values in (0, 1):
        sizes = [n + d for n in (1, 4096, 8192, 65536, 1 << 19, 1 << 21, 1 << 26) for d in (-1, 0, 1, 2049)]
        need = [lib.vren_radix_sort_scratch_bytes(n, values) for n in sorted(sizes)]
        assert need == sorted(need)
