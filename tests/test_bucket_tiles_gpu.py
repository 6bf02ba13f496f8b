"""The bucket sort of more than 2^21 pairs, whose tiles hold 15360 and 23552 pairs on 256 CUs: around the sizes where the tile
changes, in one pass (256 buckets) and in two (65536), with keys of few and of many distinct values: pairs and starts equal to
torch's stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 21) + 1, 15360 * 256 - 1, 15360 * 256, 15360 * 256 + 1, 23552 * 256, 23552 * 256 + 1,
                               (1 << 23) + 3])
@pytest.mark.parametrize("buckets,shift", [(65536, 0), (256, 0), (4096, 13)])
@pytest.mark.parametrize("distinct", [5, 1 << 32])
def test_bucket_sort_of_large_tiles(vctx, n, buckets, shift, distinct):
    g = torch.Generator(device="cuda").manual_seed(n + buckets)
    k = torch.randint(0, 1 << 32, (min(n, distinct),), device="cuda", generator=g, dtype=torch.int64)
    k = k[torch.randint(0, k.numel(), (n,), device="cuda", generator=g)]
    keys = torch.where(k >= 1 << 31, k - (1 << 32), k).to(torch.int32)
    pairs = torch.stack([keys, torch.arange(n, dtype=torch.int32, device="cuda")], dim=1).contiguous()
    out = torch.full_like(pairs, -1)
    starts = torch.full((buckets,), -1, dtype=torch.int32, device="cuda")
    vctx.bucket_sort(pairs, n, out, starts, buckets, shift)
    bucket = (k >> shift) & (buckets - 1)
    ordered, order = torch.sort(bucket, stable=True)
    want = torch.searchsorted(ordered, torch.arange(buckets, device="cuda", dtype=torch.int64)).to(torch.int32)
    assert torch.equal(out, pairs[order])
    assert torch.equal(starts, want)
