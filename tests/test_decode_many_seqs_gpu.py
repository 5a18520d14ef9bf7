"""Split decode attention where the partials pass 4 GiB: 65,536 sequences of 128 query heads over 8 KV
heads (65,792 work entries a head). The longer sequences, whose pieces are merged from those partials,
against the same sequences in a call of their own, within the bf16 tolerance (other pieces, another
order of the sums). The sequences share a few cache slots and one q row stride, so that only the
workspace is large."""

import ctypes

import pytest
import torch

from helpers import assert_attn_close, bf16_np, say

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def _decode(lib, native, q, q_sb, cache, lens, slots, dev):
    B, hq = lens.shape[0], q.shape[-2]
    nd = torch.tensor([B], dtype=torch.int32, device=dev)
    n = lib.ie_decode_attention_workspace_size(B, hq, 128)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    ws[:lib.ie_decode_attention_workspace_counts_bytes(B, hq)].zero_()
    out = torch.full((B, hq, 128), 7.0, dtype=torch.bfloat16, device=dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    i64 = ctypes.c_int64
    desc = native.KVCacheDesc.of(cache)
    fn = lib.ie_decode_attention
    fn.restype = ctypes.c_int
    rc = fn(p(q), i64(q_sb), i64(128), ctypes.c_int32(B), ctypes.c_int32(hq), ctypes.byref(desc),
            p(lens), p(slots), p(nd), ctypes.c_float(SCALE), p(out), i64(hq * 128), i64(128), p(ws),
            ctypes.c_size_t(n), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.ie_attn_last_error()
    torch.cuda.synchronize()
    return out, n


def test_partials_past_4_gib(ie, native, dev):
    lib = native.cabi()
    hq, hkv, B, L = 128, 8, 65536, 1024
    g = torch.Generator(device=dev).manual_seed(51)
    cache = ie.make_layer_cache(4, hkv, L, 128, device=dev)
    cache.k.random_(-127, 128, generator=g)
    cache.v.random_(-127, 128, generator=g)
    for t in (cache.k_scale, cache.v_scale):
        t.uniform_(0.005, 0.02, generator=g)
    q = torch.randn(1, hq, 128, generator=g, device=dev).bfloat16()
    lens = torch.zeros(B, dtype=torch.int32, device=dev)
    long = torch.tensor([0, 1, B // 2, B - 2, B - 1], device=dev)
    lens[long] = torch.tensor([700, 999, 1023, 850, 600], dtype=torch.int32, device=dev)
    slots = (torch.arange(B, device=dev, dtype=torch.int32) % 4).contiguous()
    say(f"decode B={B} {hq}/{hkv}")
    out, n = _decode(lib, native, q, 0, cache, lens, slots, dev)
    assert n > 1 << 32
    ref, _ = _decode(lib, native, q, 0, cache, lens[long].contiguous(), slots[long].contiguous(), dev)
    assert_attn_close(bf16_np(out[long]), bf16_np(ref), "sequences of several pieces")
    one = out[7].float()  # one token: its V row
    v = cache.v[3, :, 0].float() * cache.v_scale[3, :, 0, None]
    assert (one.view(hkv, 16, 128) - v[:, None]).abs().max() <= 2.0 ** -8 * v.abs().max()
