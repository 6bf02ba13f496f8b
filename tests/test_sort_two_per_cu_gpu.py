"""The radix sort where the default tile changes above one tile per CU (23552 * 256 keys on 256 CUs; with values also
20971520), last tiles of one key, a few and all but one included: equal to torch's stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [15360 * 256, 23552 * 256, 23552 * 256 + 1, 15360 * 400 + 1, 15360 * 400 - 1, 7000003,
                               20971520, 20971521])
@pytest.mark.parametrize("values", [True, False])
@pytest.mark.parametrize("begin,end,distinct", [(0, 32, 1 << 32), (3, 14, 5)])
def test_sort_above_one_tile_per_cu(vctx, n, values, begin, end, distinct):
    g = torch.Generator(device="cuda").manual_seed(n)
    k = torch.randint(0, 1 << 32, (min(n, distinct),), device="cuda", generator=g, dtype=torch.int64)
    k = k[torch.randint(0, k.numel(), (n,), device="cuda", generator=g)]
    keys = torch.where(k >= 1 << 31, k - (1 << 32), k).to(torch.int32)
    vals = torch.arange(n, dtype=torch.int32, device="cuda")
    order = torch.sort((k >> begin) & ((1 << (end - begin)) - 1), stable=True).indices
    want_keys, want_vals = keys[order], vals[order]
    scratch = torch.empty(vctx.radix_sort_scratch_bytes(n, values), dtype=torch.uint8, device="cuda")
    vctx.radix_sort(keys, vals if values else None, n, scratch, begin, end)
    assert torch.equal(keys, want_keys)
    assert not values or torch.equal(vals, want_vals)
