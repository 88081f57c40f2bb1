"""Banded soft DTW with helper waves (parts of at most four stripes): value, marginals and
temperature gradient equal the single-wave form (D2P_AMD_DTW_HELPERS=0) bit for bit,
the zeros off the band included, over bands that start and end within chunks and rows,
ragged lengths, empty elements, split parts and rows of every alignment."""
import numpy as np
import pytest
import torch

import d2p_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L1,L2,band,parts,ragged", [
    (2, 64, 64, 1, 0, False), (3, 65, 130, 5, 0, True), (2, 256, 256, 16, 0, False),
    (3, 250, 311, 64, 0, True), (2, 700, 640, 33, 3, False), (3, 512, 1024, 8, 2, True),
    (1, 1000, 90, 16, 4, False), (2, 130, 2, 1, 0, False), (2, 300, 300, 4000, 2, True),
])
def test_banded_helpers_bit_identical(cuda, monkeypatch, B, L1, L2, band, parts, ragged):
    if parts:
        monkeypatch.setenv("D2P_AMD_SPLIT", str(parts))
    g = np.random.default_rng(L1 * L2 + band)
    c = torch.from_numpy(g.random((B, L1, L2), dtype=np.float32)).to(cuda)
    lengths = None
    if ragged:
        n = np.stack([g.integers(1, L1 + 1, B), g.integers(1, L2 + 1, B)], 1).astype(np.int32)
        n[0] = L1, L2
        n[-1, 1] = 0
        lengths = torch.from_numpy(n).to(cuda)
    out = {}
    for flag in ("1", "0"):
        monkeypatch.setenv("D2P_AMD_DTW_HELPERS", flag)
        # (memory that the marginals may get: not zero by chance)
        torch.full((B, L1, L2), 7.0, device=cuda)
        out[flag] = [t.clone() for t in d2p_amd.soft_dtw_with_grads(c, 0.5, lengths, band)]
    for a, b in zip(out["1"], out["0"]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("helpers", ["0", "1"])
@pytest.mark.parametrize("L1,L2", [(1, 1), (1, 40), (40, 1), (33, 40), (40, 33), (7, 70), (129, 9),
                                   (66, 13), (64, 16), (20, 131)])
@pytest.mark.parametrize("band", [0, 1, 2, 5, 16, 1000])
def test_marginals_are_positive_in_the_band_alone(cuda, monkeypatch, L1, L2, band, helpers):
    # all paths alike: a cell's marginal is its share of the paths, 0 off the band
    # (|j - i L2 / L1| <= bandwidth in 32-bit arithmetic, as the oracle has it) and where no path
    # inside it passes
    monkeypatch.setenv("D2P_AMD_DTW_HELPERS", helpers)
    c = np.zeros((2, L1, L2), np.float32)
    want = O.get("oracle64").soft_dtw(c[:1].astype(np.float64), 1.0, None, band)[1]
    assert not ((want > 0) & (want < 1e-30)).any()
    torch.full((2, L1, L2), 7.0, device=cuda)
    got = d2p_amd.soft_dtw_with_grads(torch.from_numpy(c).to(cuda), 1.0, None, band)[1]
    assert np.array_equal(got.cpu().numpy() > 0, np.broadcast_to(want > 0, c.shape))
