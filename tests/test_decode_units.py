"""The decode launch's work entries against the workspace that is reserved for them, on the host: at
every GQA ratio from 1 to 16 and for batches on both sides of every target, the partials of the entries
fit ie_decode_attention_workspace_size."""

import pytest

BATCHES = sorted({1, 2, 300, 1000, 1024} | {c + d for c in (32, 42, 64, 85, 102, 128, 170, 256, 341, 512,
                                                            1024) for d in (-1, 0, 1)})


@pytest.mark.parametrize("hkv", [1, 2, 3, 4, 5, 7, 8, 12, 16, 32])
def test_entries_fit_the_workspace(native, hkv):
    lib = native.cabi()
    for ratio in range(1, 17):
        hq = ratio * hkv
        for b in BATCHES:
            units = lib.ie_decode_attention_units(b, hq, hkv)
            assert units > 0
            entries = lib.ie_decode_attention_grid(b, units)
            counts = lib.ie_decode_attention_workspace_counts_bytes(b, hq)
            need = counts + hq * entries * 130 * 4
            assert b <= entries, (hq, hkv, b)
            assert need <= lib.ie_decode_attention_workspace_size(b, hq, 128), (hq, hkv, b, units)
            if ratio == 2:
                assert units == hkv
    assert lib.ie_decode_attention_units(4, 3, 2) == 0
