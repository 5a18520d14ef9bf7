"""The row-major gate/up GEMM in paired tiles (three 8-column tiles per workgroup, taken where it
leaves the busiest CU fewer columns) against the reordered weight's launches, whose result bits at an
even width are those of the separate-tile row-major form: the same bits, at row counts around the
16-row tiles, plain and with the RMSNorm inside, for column counts that do and do not divide into
24-column workgroups. And the 8-row form through LDS stages: against float64, and bit for bit against
the form without them (which weights of more row blocks than CUs take)."""

import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu


def _mats(dev, M, N, K, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    return x, (0.05 * torch.randn(N, K, generator=g, device=dev)).bfloat16()


@pytest.mark.parametrize("M,nt", [(1, 1), (15, 2), (16, 1), (17, 1), (17, 2), (32, 1), (32, 2),
                                  (33, 1), (48, 1)])
@pytest.mark.parametrize("N,K", [(12288, 2048), (12288, 512), (12288 + 128, 1024)])
def test_row_pairs_bits(ie, dev, M, N, K, nt):
    say(f"gate/up {N}x{K} M={M} nt={nt}")
    x, w = _mats(dev, M, N, K, 91)
    sw = ie.swizzle_weight(w, 2 * nt, gate_up=True)
    a = ie.skinny_matmul_silu_mul(x, w, nt)
    b = ie.skinny_matmul_silu_mul(x, sw, 2 * nt, swizzled=True)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    ops = torch.ops.ie
    a = ops.skinny_matmul_norm(x, w, nt, True, 1e-6, False, False)
    b = ops.skinny_matmul_norm(x, sw, 2 * nt, True, 1e-6, True, False)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(6144, 1024), (2304, 512), (9216, 2048), (24576, 256)])
def test_row_pairs_bits_at_other_widths(ie, dev, M, N, K):
    """Widths where 24-column workgroups replace 32-column ones (n_tiles 2)."""
    say(f"gate/up {N}x{K} M={M}")
    x, w = _mats(dev, M, N, K, 93)
    a = ie.skinny_matmul_silu_mul(x, w, 2)
    b = ie.skinny_matmul_silu_mul(x, ie.swizzle_weight(w, 4, gate_up=True), 4, swizzled=True)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("K", [512, 2048, 6144])
def test_eight_row_stages_bits(ie, dev, M, K):
    """The first rows of a weight alone (one 8-row block per CU at most: through the stages) and as part
    of one of twice as many blocks as CUs (without): the same bits, plain, with the RMSNorm and with the
    residual add; x rows of a wider buffer."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    few, many = 8 * cus, 16 * cus
    say(f"8-row tiles M={M} K={K}")
    x, w = _mats(dev, M, many, K, 94)
    wide = torch.randn(M, K + 64, device=dev).bfloat16()
    wide[:, :K] = x
    x = wide[:, :K]
    ops = torch.ops.ie
    for f in (lambda w, n: ie.skinny_matmul(x, w, 0),
              lambda w, n: ops.skinny_matmul_norm(x, w, 0, False, 1e-6, False, False),
              lambda w, n: ops.skinny_matmul_residual_(x, w, 0, res[:, :n].contiguous(), False,
                                                       False)):
        res = torch.randn(M, many, device=dev).bfloat16()
        a, b = f(w[:few], few), f(w, many)
        torch.cuda.synchronize()
        assert torch.equal(a.view(torch.int16), b[:, :few].contiguous().view(torch.int16))


@pytest.mark.parametrize("M", [1, 16, 17, 40, 64])
@pytest.mark.parametrize("N,K", [(2048, 6144), (2048, 2048), (16, 512), (4096, 512), (48, 768)])
def test_eight_row_tiles(ie, dev, M, N, K):
    """K = 768 leaves no whole 64-column batch per wave: the form without stages. Against float64:
    fp32 sums of K bf16 products, then one bf16 rounding (2^-9), each product's error at most
    K 2^-24 of the sum of magnitudes."""
    x, w = _mats(dev, M, N, K, 92)
    got = ie.skinny_matmul(x, w, 0).double()
    ref = x.double() @ w.double().T
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().T) * (K * 2.0 ** -24)
    assert ((got - ref).abs() <= bound).all()
