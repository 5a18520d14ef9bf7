"""fused_norm_rope_prefill on 16-byte aligned rows (16 lanes per head row) against the form for any
alignment (one wave per row group, the one the oracle tests pin as well), bit for bit: head counts
that fill a wave's row groups, leave a remainder of rows or of groups or mix q and k in a group, token
counts on both sides of the groups-per-wave rule (one, three or six groups of four rows a wave), rows
of very different magnitude, and rows of zeros."""

import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv", [(16, 8), (2, 1), (7, 7), (5, 1), (40, 8), (1, 1)])
@pytest.mark.parametrize("n", [1, 3, 515, 4097])
def test_aligned_rows_equal_unaligned_rows(ie, dev, hq, hkv, n):
    _check(ie, dev, hq, hkv, n)


# 3, 4, 5 and 10 groups (three a wave, the last wave's all there, one, two and one), 13, 14 and 17 (six
# a wave, one, two and five in the last), on both sides of 98,304 rows
@pytest.mark.parametrize("hq,hkv", [(8, 4), (8, 5), (16, 4), (32, 8), (44, 8), (48, 6), (64, 4)])
@pytest.mark.parametrize("rows", [90_000, 98_304, 110_001])
def test_groups_per_wave(ie, dev, hq, hkv, rows):
    _check(ie, dev, hq, hkv, -(-rows // (hq + hkv)))


def _check(ie, dev, hq, hkv, n):
    say(f"norm rope {hq}+{hkv} heads, {n} tokens")
    g = torch.Generator(device=dev).manual_seed(81)
    h = hq + hkv
    x = torch.randn(n, h, 128, generator=g, device=dev)
    x *= 10.0 ** torch.randint(-6, 6, (n, h, 1), generator=g, device=dev)
    x[n // 2, h - 1] = 0.0
    x = x.bfloat16()
    w = (1 + 0.3 * torch.randn(2, 128, generator=g, device=dev)).bfloat16()
    ang = 1000 * torch.rand(n, 1, 64, generator=g, device=dev)
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    wide = torch.empty(n, h * 128 + 3, dtype=torch.bfloat16, device=dev)  # rows 2 bytes off
    odd = wide[:, 1:h * 128 + 1].view(n, h, 128).copy_(x)
    got = ie.fused_norm_rope_prefill(x[:, :hq], x[:, hq:], w[0], w[1], cos, sin, 1e-6)
    ref = ie.fused_norm_rope_prefill(odd[:, :hq], odd[:, hq:], w[0], w[1], cos, sin, 1e-6)
    torch.cuda.synchronize()
    for a, b in zip(got, ref):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
