"""tune_linear's choice of the gate/up tile width, whose two values differ in result bits: timing noise
between equal times does not change it, a real difference does. The timer is replaced, nothing is
launched."""

import pytest
import torch


@pytest.mark.parametrize("t1,t2,want", [(12.0, 12.0, 2), (11.9, 12.1, 2), (12.1, 11.9, 2),
                                        (11.75, 12.0, 2), (16.3, 12.4, 2), (10.9, 13.0, 1)])
def test_equal_times_give_one_width(ie, monkeypatch, t1, t2, want):
    K = ie.kernels
    N, D, M = 128, 256, 32
    order = []

    def time(fns):  # the library, skinny n_tiles 0, 1, 2, 4, then gate/up widths 1 and 2 twice each
        order.append(None)
        times = {1: 30.0, 6: t1, 7: 1.2 * t1, 8: 1.1 * t2, 9: t2}
        return times.get(len(order), 20.0)

    monkeypatch.setattr(K, "_graph_time", time)
    monkeypatch.setattr(K, "swizzle_weight", lambda w, nt, gate_up=False: w)
    for name in ("use_skinny", "use_skinny_glu", "use_skinny_swz", "use_skinny_glu_swz"):
        monkeypatch.setattr(K, name, {})
    w = torch.zeros(N, D).bfloat16()
    monkeypatch.setattr(torch.Tensor, "clone", lambda self, *a, **k: self)
    K.tune_linear([w], [M])
    assert K.use_skinny_glu[(N, D, M)] == want
