"""The decode kernel's tiles at their edges: a wave's block holds 32 tokens, a workgroup round 32 per
wave (8-, 4-, 2- and one-wave workgroups by batch and heads), the 16 columns of a tile hold a KV head's query
heads. Sequence lengths around those sizes at odd and full ratios, workgroups of every width, the
few-KV-head layouts whose entries are cut to the workspace, `out` rows that take no 8-byte store, and
V scales that leave the fp16 window mid-sequence; against the oracle with the bf16 tolerance."""

import numpy as np
import pytest
import torch

from helpers import assert_attn_close, bf16_np, cache_np, say
from oracle import attention as oat

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5
EDGES = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 160, 255, 257, 640, 1023, 4097]


def _ref(wl):
    return oat.decode_attention(bf16_np(wl.q), cache_np(wl.cache), wl.cached_lens.numpy(),
                                wl.slot_ids.numpy(), int(wl.num_decoding[0]), SCALE)


def _run(ie, wl, dev, out=None):
    g = wl.to(dev)
    out = ie.decode_attention(g.q, g.cache, g.cached_lens, g.slot_ids, g.num_decoding, SCALE,
                              out=out)
    torch.cuda.synchronize()
    return bf16_np(out)


@pytest.mark.parametrize("hq,hkv", [(8, 8), (16, 8), (24, 8), (7, 1), (64, 4), (16, 2), (16, 1)])
def test_lengths_at_tile_edges(ie, workloads, dev, hq, hkv):
    say(f"decode edges {hq}/{hkv}")
    wl = workloads.decode_workload(EDGES, seed=71, hq=hq, hkv=hkv)
    assert_attn_close(_run(ie, wl, dev), _ref(wl), f"{hq}/{hkv}")


@pytest.mark.parametrize("batch,hq,hkv", [(65, 16, 8), (129, 16, 8), (70, 64, 8), (140, 32, 8),
                                          (300, 12, 4), (300, 64, 4)])
def test_narrow_workgroups(ie, workloads, dev, batch, hq, hkv):
    say(f"decode B={batch} {hq}/{hkv}")
    ctx = [EDGES[i % 15] for i in range(batch)]
    wl = workloads.decode_workload(ctx, seed=72, hq=hq, hkv=hkv)
    assert_attn_close(_run(ie, wl, dev), _ref(wl), f"B={batch} {hq}/{hkv}")


@pytest.mark.parametrize("batch,heads", [(129, 16), (256, 16), (257, 16), (257, 8), (100, 7), (65, 32)])
def test_batches_past_a_target_at_ratio_1(ie, workloads, dev, batch, heads):
    """Batches that pass the largest target of as many units as KV heads: the entries are cut to the
    workspace, which is sized by the query heads alone."""
    say(f"decode B={batch} {heads}/{heads}")
    ctx = [EDGES[i % 15] for i in range(batch)]
    wl = workloads.decode_workload(ctx, seed=77, hq=heads, hkv=heads)
    out = _run(ie, wl, dev)
    assert_attn_close(out, _ref(wl), f"B={batch} {heads}/{heads}")
    g = wl.to(dev)
    planned = ie.decode_attention(g.q, g.cache, g.cached_lens, g.slot_ids, g.num_decoding, SCALE,
                                  plan=ie.decode_plan(g.cached_lens, g.num_decoding, batch, heads,
                                                      heads))
    assert np.array_equal(bf16_np(planned), out)


def test_out_rows_without_8_byte_alignment(ie, workloads, dev):
    wl = workloads.decode_workload([33, 2000, 700], seed=73, hq=32, hkv=8)
    buf = torch.full((3, 32, 131), 5.0, dtype=torch.bfloat16, device=dev)
    out = buf[:, :, 1:129]
    assert_attn_close(_run(ie, wl, dev, out), _ref(wl), "odd out rows")
    assert (buf[:, :, 0] == 5.0).all() and (buf[:, :, 129:] == 5.0).all()


@pytest.mark.parametrize("hq,hkv", [(16, 8), (32, 8)])
def test_v_scales_that_move(ie, workloads, dev, hq, hkv):
    """V's scales rise by 2^12 and fall by 2^14 along the sequence (the exponent under which P times
    scale is held in fp16 has to follow): outputs relative to the largest of them."""
    wl = workloads.decode_workload([1500, 90, 3000], seed=74, hq=hq, hkv=hkv)
    vs = wl.cache.v_scale
    vs[:, :, 200:700] *= 2.0 ** 12
    vs[:, :, 700:] *= 2.0 ** -2
    got, ref = _run(ie, wl, dev), _ref(wl)
    scale = np.abs(ref).max(axis=-1, keepdims=True)
    assert_attn_close(got / scale, ref / scale, "moving V scales", rel=False)


@pytest.mark.parametrize("hq,hkv,B,waves", [
    (64, 4, 300, 1), (128, 8, 140, 1),  # q's rows over the second stage: one wave, over 8 heads
    (64, 8, 150, 1), (16, 8, 140, 1),   # one wave, q's rows beside the stages
    (64, 4, 520, 2), (64, 8, 100, 2),
    (64, 8, 12, 4), (40, 8, 5, 4),
    (64, 4, 20, 8), (16, 1, 4, 8), (12, 4, 30, 8)])
def test_fused_form_in_every_width(ie, native, dev, hq, hkv, B, waves):
    """decode_attention_rope in workgroups of every number of waves: the same cache, bit for bit, as
    fused_rope_kv_decode then decode_attention, and the same output within the tolerance (there q
    comes from memory and the new token from the cache). Lengths at which every wave has blocks of
    both its stages."""
    L = 400 if waves <= 2 else 6000
    lib = native.cabi()
    units = lib.ie_decode_attention_units(B, hq, hkv)
    width = {lib.ie_decode_attention_max_splits(units) // w: w for w in (1, 2, 4)}
    named = min(8, width.get(lib.ie_decode_attention_target(B, units), 0) * units // hkv)
    assert named == waves, f"the launch has {named}-wave workgroups"
    g = torch.Generator().manual_seed(75)
    qkv = torch.randn(B, (hq + 2 * hkv) * 128, generator=g).bfloat16().to(dev)
    q, k, v = (x.view(B, -1, 128) for x in qkv.split([hq * 128, hkv * 128, hkv * 128], -1))
    w = (1 + 0.2 * torch.randn(2, 128, generator=g)).bfloat16().to(dev)
    lens = torch.randint(0, L - 1, (B,), generator=g, dtype=torch.int32).to(dev)
    slots = torch.randperm(B, generator=g).int().to(dev)
    ang = lens[:, None, None].float() * (1e6 ** (-torch.arange(0, 128, 2, device=dev) / 128.0))
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    nd = torch.tensor([B], dtype=torch.int32, device=dev)
    caches = []
    for _ in range(2):
        c = ie.make_layer_cache(B, hkv, L, 128, device=dev)
        gc = torch.Generator(device=dev).manual_seed(76)
        c.k.copy_(torch.randint(-127, 128, c.k.shape, generator=gc, device=dev))
        c.v.copy_(torch.randint(-127, 128, c.v.shape, generator=gc, device=dev))
        c.k_scale.copy_(torch.rand(c.k_scale.shape, generator=gc, device=dev) * 0.02)
        c.v_scale.copy_(torch.rand(c.v_scale.shape, generator=gc, device=dev) * 0.02)
        caches.append(c)
    out = ie.decode_attention_rope(q, k, v, w[0], w[1], cos, sin, slots, caches[0], lens, nd, 1e-6,
                                   SCALE)
    qn = ie.fused_rope_kv_decode(q, k, v, w[0], w[1], cos, sin, slots, caches[1], lens, nd, 1e-6)
    ref = ie.decode_attention(qn, caches[1], lens, slots, nd, SCALE)
    torch.cuda.synchronize()
    for name in ("k", "v", "k_scale", "v_scale"):
        assert torch.equal(getattr(caches[0], name), getattr(caches[1], name)), name
    assert_attn_close(bf16_np(out), bf16_np(ref), "fused against two launches")


def test_output_of_its_own(ie, workloads, dev):
    """Without `out`: a contiguous [B, Hq, D] tensor whatever q's strides, that requires no gradient
    whatever q does, with the values that a given `out` gets."""
    wl = workloads.decode_workload([5, 300, 70], seed=76)
    g = wl.to(dev)
    wide = torch.randn(3, g.q.shape[1] + 4, 128, device=dev).bfloat16()
    q = wide[:, 2:-2]
    q.copy_(g.q)
    args = (g.cache, g.cached_lens, g.slot_ids, g.num_decoding, SCALE)
    out = torch.empty_like(g.q)
    ie.decode_attention(g.q, *args, out=out)
    own = ie.decode_attention(q.requires_grad_(), *args)
    assert own.is_contiguous() and own.shape == g.q.shape and own.dtype == g.q.dtype
    assert not own.requires_grad
    assert torch.equal(own, out)
