"""Into how many time segments the stand-alone scans of 2-byte elements cut a sequence (scan_segments, csrc/api.hip): read off the
workspace, which holds the segments' records.  On the CPU."""
import ctypes

import pytest
import torch

from hdla_hip import _lib


def _segments(K, V, lanes, chunks, bwd, N=1, dtype=torch.bfloat16):
    def need(**kw):
        d = _lib.make_dims(1, 16 * chunks * N, lanes // N, K, V, 2, N, dtype, dtype, 1.0, None, **kw)
        if N > 1:
            d.cu_seqlens = 256                                  # never read on the host
        return _lib.load().hdla_workspace_bytes(ctypes.byref(d), int(bwd))
    return [n for n in range(1, 33) if need(segments=n) == need()]


# the fastest of 1, 4, 8, 16 and 32 segments, with the next one's time over its own
@pytest.mark.parametrize("K,V,lanes,chunks,bwd,want", [
    (128, 128, 2, 97, False, 8),        # 1.08
    (128, 128, 8, 64, False, 1), (128, 128, 8, 64, True, 1),        # 1.00, 1.11
    (128, 128, 8, 97, False, 8), (128, 128, 8, 97, True, 1),        # 1.10, 1.02
    (128, 128, 24, 97, False, 1),       # 1.34
    (128, 128, 16, 97, False, 1), (128, 128, 16, 97, True, 1),      # 1.01, 1.17
    (128, 128, 8, 313, False, 8),       # 1.10
    (64, 128, 4, 64, False, 8),         # 1.08
    (64, 128, 8, 64, True, 1),          # 1.12
    (128, 64, 2, 128, True, 8),         # 1.09
])
def test_the_fastest_is_chosen(K, V, lanes, chunks, bwd, want):
    assert _segments(K, V, lanes, chunks, bwd) == [want]


@pytest.mark.parametrize("bwd,most", [(False, 128), (True, 64)])
@pytest.mark.parametrize("K,V", [(64, 128), (128, 64), (128, 128)])
def test_bounds(K, V, bwd, most):
    for lanes in (1, 2, 3, 5, 12, 33, 64, 129, 4096):
        for chunks in (0, 1, 3, 17, 1000, 100000):
            if lanes * chunks > 1 << 20:
                continue
            n = _segments(K, V, lanes, chunks, bwd)[0]          # (of many lanes more are taken for fewer)
            assert n in (1, 4, 8, 16, 32) and (n == 1 or lanes * n <= most) and (chunks > 17 or n == 1)


def test_packed_sequences_are_expected_to_be_of_unequal_lengths():
    """Two sequences of 8 heads: a longest one of 1.6 times the average makes segments worth their launches (1.10)."""
    assert _segments(128, 64, 16, 66, False) == [1] and _segments(128, 64, 16, 66, False, N=2)[0] > 1
    for lanes, chunks in ((2, 97), (8, 313), (64, 1000), (2, 1)):
        for bwd in (False, True):
            assert _segments(128, 128, lanes, chunks, bwd, N=2)[0] >= _segments(128, 128, lanes, chunks, bwd)[0]
