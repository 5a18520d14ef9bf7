"""The decode calls under tracing: with fake tensors (no device, nothing launched) they give a fake
output of q's shape, with and without an output of the caller's, and one recorded call each."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx


def _args(ie, b=3, hq=16, hkv=8):
    bf = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    i = torch.zeros(b, dtype=torch.int32, device="cuda")
    nd = torch.zeros(1, dtype=torch.int32, device="cuda")
    c = ie.make_layer_cache(b, hkv, 64, 128, device="cuda")
    wide = bf(b, hq + 2, 128)
    return wide[:, 1:-1], bf(b, hkv, 128), bf(128), bf(b, 1, 64), i, nd, c


@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("rope", [True, False])
def test_fake_tensors(ie, own, rope):
    ie.kernels.ops()
    with FakeTensorMode(allow_non_fake_inputs=True):
        q, k, w, cs, i, nd, c = _args(ie)
        out = None if own else torch.empty(3, 16, 128, dtype=q.dtype, device="cuda")

        def call(q):
            if rope:
                return ie.decode_attention_rope(q, k, k, w, w, cs, cs, i, c, i, nd, 1e-6, 0.1, out=out)
            return ie.decode_attention(q, c, i, i, nd, 0.1, out=out)

        got = call(q)
        assert got.shape == (3, 16, 128) and got.dtype == q.dtype and got.device.type == "cuda"
        assert got.is_contiguous()
        ops = [n.target for n in make_fx(call)(q).graph.nodes if "decode" in str(n.target)]
        assert len(ops) == 1
