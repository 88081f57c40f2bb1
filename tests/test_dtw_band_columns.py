"""A banded row's valid columns as an interval (band_columns in dtw_internal.hip.h): the
interval's ends, found from the unrounded ones, against the band test of every column
(|j - i L2 / L1| <= bandwidth in 32-bit arithmetic), emulated with numpy."""
import numpy as np
import pytest

f32 = np.float32


def _in_band(ej, j, bw):
    return np.abs(f32(j) - ej) <= bw


def _columns(ej, bw, L2):
    lo = max(int(np.floor(max(ej - bw, f32(-8)))) - 3, 0)
    hi = min(int(np.ceil(min(ej + bw, f32(L2) + f32(8)))) + 2, L2 - 1)
    for _ in range(8):
        lo += not _in_band(ej, lo + 1, bw)
        hi -= not _in_band(ej, hi + 1, bw)
    return lo, max(hi - lo + 1, 0)


@pytest.mark.parametrize("L1,L2", [(1, 1), (1, 300), (300, 1), (64, 65), (333, 1000),
                                   (4096, 4096), (7, 262080), (262080, 997)])
def test_band_columns_are_the_in_band_cells(L1, L2):
    rng = np.random.default_rng(L1 + L2)
    rows = np.unique(np.r_[1, L1, rng.integers(1, L1 + 1, 12)])
    j = np.arange(1, L2 + 1)
    for bandwidth in (0, 1, 2, 16, 64, 1 << 20, (1 << 31) - 1):
        bw = f32(bandwidth)
        for i in rows:
            ej = f32(int(i) * L2) / f32(L1)
            want = np.flatnonzero(np.abs(j.astype(f32) - ej) <= bw)
            lo, n = _columns(ej, bw, L2)
            assert n == len(want)
            if n:
                assert lo == want[0] and lo + n - 1 == want[-1]
