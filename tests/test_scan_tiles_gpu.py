"""The exclusive scan around the tile sizes it chooses from (one workgroup up to 32768 elements, tiles of 16384 up to 2^21
elements, then of 32768, and of 65536 above 2^23 elements in segments of 2^18 and more): last tiles of one element to all but one, segments that start on any
4-byte boundary, in place; equal to a 64-bit prefix sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,blocks", [
    (16385, 1), (32767, 3), (32768, 2), (32769, 3), (65535, 1), (65537, 5), (98305, 1), ((1 << 18) - 1, 40),
    (1 << 18, 32), (1 << 21, 1), ((1 << 21) + 1, 1), (32769, 64), (49153, 50), (1 << 18, 33), ((1 << 18) + 1, 40), ((1 << 19) + 2, 17), (1 << 23, 1), ((1 << 23) + 1, 1),
    ((1 << 23) + 65535, 1), (3000003, 3)])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_scan_tiles(vctx, n, blocks, shift):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(-1 << 31, 1 << 31, (n * blocks + shift + 4,), device="cuda", generator=g, dtype=torch.int64).to(torch.int32)
    body = x[shift:shift + n * blocks]
    wide = body.view(blocks, n).long()
    want = (torch.cumsum(wide, 1) - wide).to(torch.int32).reshape(-1)
    out = torch.full_like(x, 7)
    vctx.exclusive_scan_u32(body, out[shift:], n, blocks)
    assert torch.equal(out[shift:shift + n * blocks], want)
    assert bool((out[:shift] == 7).all()) and bool((out[shift + n * blocks:] == 7).all())
    after = x[shift + n * blocks:].clone()
    vctx.exclusive_scan_u32(body, body, n, blocks)
    assert torch.equal(body, want) and torch.equal(x[shift + n * blocks:], after)
