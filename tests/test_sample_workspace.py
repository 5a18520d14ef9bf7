"""ie_sample_workspace_size on the host: it grows with the batch and with the vocabulary, so that a
workspace made for the largest of either serves the smaller ones too."""

import ctypes

import pytest


@pytest.mark.parametrize("vocab", [1, 2048, 2049, 4096, 4097, 151_669, 151_936])
def test_size_never_falls(native, vocab):
    size = native.cabi().ie_sample_workspace_size
    size.restype = ctypes.c_size_t
    at = lambda b, v: size(ctypes.c_int32(b), ctypes.c_int64(v))
    assert at(0, vocab) == 0
    batches = list(range(1, 80)) + [255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 4096]
    sizes = [at(b, vocab) for b in batches]
    assert sizes[0] > 0 and all(a <= b for a, b in zip(sizes, sizes[1:]))
    assert all(at(b, vocab) <= at(b, vocab + 1) for b in batches)
