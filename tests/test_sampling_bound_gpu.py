"""sample at tau != 0 where entries that cannot win are not drawn: the tokens are still the oracle's,
for logits whose winner is a candidate, comes out of the bulk by its noise alone, or is among equal
entries; for rows with -inf entries (masked vocabularies) up to all of them; for vocabularies around
the block sizes (2,048 and 4,096 entries) and batches on both sides of the block-size rule; for
candidate counts around the list's capacity (3/4 of a block); and for a negative tau."""

import numpy as np
import pytest
import torch

from helpers import say
from oracle import sampling as osm

pytestmark = pytest.mark.gpu


def _check(ie, x, tau, s0, dev, dtype=torch.bfloat16):
    x = x.to(dtype)
    seed = torch.tensor([s0], dtype=torch.int64, device=dev)
    tok = ie.sample(x.to(dev), tau, seed).cpu().numpy()
    ref, nxt = osm.sample(x.float().numpy(), tau, s0)
    say(f"tau={tau} {tuple(x.shape)} {dtype}")
    assert np.array_equal(tok, ref), np.nonzero(tok != ref)[0][:8]
    assert int(seed.item()) == nxt


@pytest.mark.parametrize("V", [1, 7, 2047, 2048, 2049, 4096, 4097, 12289])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_vocabularies_around_the_blocks(ie, dev, V, dtype):
    g = torch.Generator().manual_seed(V)
    for B in (3, 700):  # 2,048-entry blocks; 4,096-entry ones from 1,024 workgroups
        _check(ie, 3 * torch.randn(B, V, generator=g), 0.9, V, dev, dtype)


@pytest.mark.parametrize("spread,lift,tau", [(2.0, 14.0, 0.7), (2.0, 14.0, 1.0), (2.0, 0.0, 1.0),
                                             (0.0, 0.0, 1.0), (8.0, 0.0, 0.1), (1.0, 30.0, 2.0),
                                             (2.0, 6.0, -0.5)])
def test_bulk_and_candidates(ie, dev, spread, lift, tau):
    g = torch.Generator().manual_seed(11)
    for B, V in ((2, 151_936), (40, 151_669)):
        x = spread * torch.randn(B, V, generator=g)
        x[:, torch.randint(0, V, (30,), generator=g)] += lift * torch.rand(30, generator=g)
        for s0 in (3, 2 ** 33 + 5):
            _check(ie, x, tau, s0, dev)


def test_masked_rows(ie, dev):
    g = torch.Generator().manual_seed(12)
    x = torch.randn(6, 20_000, generator=g)
    x[0, 50:] = -float("inf")
    x[1, :] = -float("inf")
    x[2, :19_999] = -float("inf")
    x[3, ::2] = -float("inf")
    x[4, 777] = float("inf")
    x[5, :] = 1.5
    for tau in (0.7, 3.0):
        _check(ie, x, tau, 21, dev)


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_candidates_around_the_list_capacity(ie, dev, extra):
    """The bound leaves every entry at 0 a candidate and none at -100: exactly n per block."""
    for B, block in ((2, 2048), (600, 4096)):
        x = torch.full((B, 2 * block), -100.0)
        x[:, : block * 3 // 4 + extra] = 0.0
        x[:, 2 * block - 5:] = 0.0
        _check(ie, x, 1.0, 31 + extra, dev)


@pytest.mark.parametrize("B", [1, 16, 17, 18, 24])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_batches_around_the_bound_launch(ie, dev, B, dtype):
    """Up to five workgroups per CU a block bounds its entries by its own largest one (17 rows of 75
    blocks are the last there on 256 CUs), above by the row's best; odd rows start unaligned."""
    g = torch.Generator().manual_seed(B)
    x = 2 * torch.randn(B, 151_937, generator=g)
    x[:, torch.randint(0, 151_937, (30,), generator=g)] += 14 * torch.rand(30, generator=g)
    _check(ie, x, 0.7, 40 + B, dev, dtype)


@pytest.mark.parametrize("V", [2 ** 28, 2 ** 28 + 4099])
@pytest.mark.parametrize("tau", [0.0, 0.7])
def test_vocabularies_past_2_28(ie, dev, V, tau):
    """Entries that no noise can lift past the one planted far above them, in the last block."""
    say(f"sample 1 x {V} tau={tau}")
    x = torch.full((1, V), -20.0, dtype=torch.bfloat16, device=dev)
    x[0, V - 3] = 30.0
    seed = torch.tensor([9], dtype=torch.int64, device=dev)
    assert int(ie.sample(x, tau, seed).item()) == V - 3
    assert int(seed.item()) == 10
