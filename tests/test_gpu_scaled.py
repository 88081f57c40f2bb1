"""The linear-domain sweeps of soft Smith-Waterman and Needleman-Wunsch (64-bit values with
an exponent per lane, factors 2^(c s) in 32 bits) against the double-precision oracle, at
the edges of their stripes, chunks, parts and launch shapes, and their hand-over of
elements whose values leave the range to the log-domain sweeps.

Tolerance: a factor's relative error is delta = 2^-23 + 2^-24 max|c s| (the 32-bit 2^x, and
the rounding of its argument).  A path of m matches multiplies m factors, whose roundings
are independent: the logarithm of a marginal is off by some sqrt(m) delta on either side of
a cell; four standard deviations of the two together are 8 sqrt(m) delta.
"""
import math

import numpy as np
import pytest
import torch

import d2p_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (B, L1, L2, temperature, gap, parts asked for (0: the library's choice), ragged)
CASES = [
    (1, 1, 1, 1.0, -1.0, 0, False),
    (2, 63, 15, 1.0, -1.0, 0, False),      # below a stripe and a chunk
    (2, 64, 16, 1.0, 0.0, 0, False),       # exactly one of each
    (3, 65, 17, 0.7, -2.0, 0, False),      # one row and one column more
    (2, 130, 1, 1.0, -1.0, 0, False),      # one column
    (2, 1, 131, 1.0, -1.0, 0, False),      # one row
    (9, 256, 90, 0.2, -0.5, 0, True),      # four stripes, lowest temperature taken
    (3, 257, 66, 1.0, -1.0, 0, True),      # five stripes: two parts
    (3, 300, 83, 1.0, -1.0, 5, True),      # parts of one stripe
    (2, 512, 203, 3.0, 1.0, 1, True),      # eight stripes in one part, a positive gap
    (300, 100, 45, 1.0, -1.0, 0, True),    # more elements than CUs: one reverse wave a stripe
    (2, 600, 40, 1.0, -1.0, 1, True),      # ten stripes: parts of at most six
    (1, 1024, 1024, 1.0, -1.0, 0, False),  # the longest taken
]


def _inputs(B, L1, L2, ragged):
    g = np.random.default_rng(1000 * L1 + L2)
    s = (1.5 * g.standard_normal((B, L1, L2))).astype(np.float32)
    if not ragged:
        return s, None
    lengths = np.stack([g.integers(0, L1 + 1, B), g.integers(0, L2 + 1, B)], 1).astype(np.int32)
    lengths[0] = L1, L2
    lengths[-1] = 0, L2
    return s, lengths


def _tol(s, m, T):
    delta = 2.0 ** -23 + 2.0 ** -24 * float(np.abs(s).max()) / T * math.log2(math.e)
    return 8.0 * math.sqrt(m) * delta


def _check(got, want, s, gaps, T, tol, glob=False):
    """Every output of the elements against the 64-bit oracle's.  tol bounds the logarithm of
    a marginal, so a sum of marginals is off by at most tol times its terms' sizes: the
    gaps are counted by such a sum (global alignment: by L1 + L2 less two for each match),
    and dS/dT = (S - sum P s - sum gaps n_gap) / T has the terms that `terms` adds up.  What is
    rounded to 32 bits at the end adds 2^-23 of itself."""
    got = [x.cpu().numpy().astype(np.float64) for x in got]
    value, post = want[0], want[1]
    assert np.all(np.abs(got[0] - value) <= T * tol + 2.0 ** -23 * np.abs(value)), (got[0], value)
    err = np.abs(got[1] - post).max()
    assert err <= tol, (err, tol)
    matches = post.sum(axis=(1, 2))
    terms = np.abs(value) + (post * np.abs(np.where(post > 0, s, 0))).sum(axis=(1, 2))
    for n, (gap, g, w) in enumerate(zip(gaps, got[2:-1], want[2:-1])):
        bound = tol * (np.abs(w) + (4 * matches + 1 if glob else 0)) + 2.0 ** -22 * np.abs(w)
        assert np.all(np.abs(g - w) <= bound + 1e-30), (n, g, w, bound)
        terms = terms + np.abs(gap) * (np.abs(w) + (4 * matches if glob else 0))
    bound = (tol + 2.0 ** -22) * terms / T
    assert np.all(np.abs(got[-1] - want[-1]) <= bound), (got[-1], want[-1], bound)


@pytest.mark.parametrize("nw", [False, True])
@pytest.mark.parametrize("B,L1,L2,T,gap,parts,ragged", CASES)
def test_scaled_sweeps_match_double_oracle(cuda, monkeypatch, B, L1, L2, T, gap, parts, ragged,
                                           nw):
    if parts:
        monkeypatch.setenv("D2P_AMD_SPLIT", str(parts))
    s, lengths = _inputs(B, L1, L2, ragged)
    op = "soft_nw" if nw else "soft_sw"
    lt = None if lengths is None else torch.from_numpy(lengths).to(cuda)
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), gap, T, lt)
    n = min(B, 9)
    idx = list(range(n - 1)) + [B - 1]
    want = getattr(O.get("oracle64"), op)(s[idx].astype(np.float64), gap, T,
                                           None if lengths is None else lengths[idx])
    _check([x[idx] for x in got], want, s[idx], (gap,), T, _tol(s, min(L1, L2), T), nw)


@pytest.mark.parametrize("nw", [False, True])
@pytest.mark.parametrize("B,L1,L2,T,gap,parts,ragged", CASES)
def test_scaled_affine_sweeps_match_double_oracle(cuda, monkeypatch, B, L1, L2, T, gap, parts,
                                                  ragged, nw):
    if parts:
        monkeypatch.setenv("D2P_AMD_SPLIT", str(parts))
    s, lengths = _inputs(B, L1, L2, ragged)
    op = "soft_nw_affine" if nw else "soft_sw_affine"
    lt = None if lengths is None else torch.from_numpy(lengths).to(cuda)
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), gap - 1.0, gap / 2,
                                               T, lt)
    n = min(B, 9)
    idx = list(range(n - 1)) + [B - 1]
    want = getattr(O.get("oracle64"), op)(s[idx].astype(np.float64), gap - 1.0, gap / 2, T,
                                          None if lengths is None else lengths[idx])
    _check([x[idx] for x in got], want, s[idx], (gap - 1.0, gap / 2), T,
           _tol(s, min(L1, L2), T), nw)


@pytest.mark.parametrize("op,gaps", [("soft_sw", (-1.0,)), ("soft_nw", (-1.0,)),
                                     ("soft_sw_affine", (-2.0, -0.5)),
                                     ("soft_nw_affine", (-2.0, -0.5))])
@pytest.mark.parametrize("L1,L2", [(40, 37), (130, 70), (300, 83)])
def test_elements_out_of_range(cuda, L1, L2, op, gaps):
    # element 1 has a factor beyond 32 bits: the log-domain sweeps compute it, whose
    # rounding is that of alpha (ulp(512), over T) along the path; element 2 is masked
    s, _ = _inputs(3, L1, L2, False)
    s[1, L1 // 2, L2 // 2] = 300.0
    s[2, :, L2 // 3:] = -1e30
    got = getattr(d2p_amd, op)(torch.from_numpy(s).to(cuda), *gaps, 1.0)
    want = getattr(O.get("oracle64"), op)(s.astype(np.float64), *gaps, 1.0, None)
    tol = _tol(np.clip(s[0], -10, 10), min(L1, L2), 1.0)
    err = np.abs(got[1].cpu().numpy() - want[1]).max(axis=(1, 2))
    assert err[0] <= tol and err[2] <= tol, err
    assert err[1] <= math.sqrt(L1 + L2) * 2.0 ** -15, err
    v = got[0].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(v - want[0]) <= 1e-5 * np.abs(want[0]) + 1e-5), (v, want[0])


@pytest.mark.parametrize("op,gaps", [("soft_sw", (-1.0,)), ("soft_nw", (-1.0,)),
                                     ("soft_sw_affine", (-2.0, -0.5)),
                                     ("soft_nw_affine", (-2.0, -0.5))])
@pytest.mark.parametrize("B,L1,L2,parts", [
    (3, 700, 90, 0),     # both: parts of at most four stripes
    (3, 300, 83, 5),     # one stripe a part
    (3, 600, 40, 1),     # log-domain sweeps of ten stripes in one workgroup
    (70, 1000, 40, 0),   # parts of eight stripes
    (300, 450, 30, 0),   # eight stripes, unsplit
    (20, 500, 66, 0),
    (3, 1000, 1, 0),
])
def test_elements_out_of_range_in_every_shape(cuda, monkeypatch, B, L1, L2, parts, op, gaps):
    # the shapes that the log-domain sweeps have for themselves; element 1 is out of range (and
    # ragged), and so is the last one
    if parts:
        monkeypatch.setenv("D2P_AMD_SPLIT", str(parts))
    s, _ = _inputs(B, L1, L2, False)
    lengths = np.full((B, 2), (L1, L2), np.int32)
    lengths[1] = L1 - 70, L2 - L2 // 3
    for b in (1, B - 1):
        s[b, L1 // 2, L2 // 2] = 300.0
    x, lt = torch.from_numpy(s).to(cuda), torch.from_numpy(lengths).to(cuda)
    f = getattr(d2p_amd, op + "_with_grads")
    got = f(x, *gaps, 1.0, lt)
    idx = [0, 1, B - 1]
    want = getattr(O.get("oracle64"), op)(s[idx].astype(np.float64), *gaps, 1.0, lengths[idx])
    tol = _tol(np.clip(s[0], -10, 10), min(L1, L2), 1.0)
    for i, b in enumerate(idx):
        # (alpha's rounding, ulp(512) and over T, along the path)
        _check([v[b:b + 1] for v in got], [w[i:i + 1] for w in want], s[b:b + 1], gaps, 1.0,
               tol if b == 0 else math.sqrt(L1 + L2) * 2.0 ** -15, "nw" in op)
    for _ in range(3):
        again = f(x, *gaps, 1.0, lt)
        for a, b in zip(got, again):
            assert torch.equal(a, b)


@pytest.mark.parametrize("op,gaps", [("soft_sw", (-1.0,)), ("soft_nw", (-1.0,)),
                                     ("soft_sw_affine", (-2.0, -0.5)),
                                     ("soft_nw_affine", (-2.0, -0.5))])
def test_elements_out_of_range_in_a_graph(cuda, op, gaps):
    # a replay has the progress words, and the epochs in them, of the one before
    f = getattr(d2p_amd, op + "_with_grads")
    inputs = []
    for seed in range(4):
        s = np.random.default_rng(seed).standard_normal((3, 700, 90)).astype(np.float32)
        s[seed % 3, 350, 40] = 300.0
        inputs.append(torch.from_numpy(s).to(cuda))
    want = [f(x, *gaps, 1.0, None) for x in inputs]
    static = inputs[0].clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = f(static, *gaps, 1.0, None)
    for i in (0, 1, 2, 3, 3, 1):
        static.copy_(inputs[i])
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want[i]):
            assert torch.equal(a, b), i


@pytest.mark.parametrize("B,L1,L2", [(300, 130, 66), (40, 300, 200)])
def test_affine_calls_repeat_bit_for_bit(cuda, B, L1, L2):
    # a wave reads its first chunks' scores only once they have arrived: workgroups that
    # start on LDS with other contents (a NaN element's, say) give the same results
    s, _ = _inputs(B, L1, L2, False)
    x = torch.from_numpy(s).to(cuda)
    want = d2p_amd.soft_sw_affine_with_grads(x, -2.0, -0.5, 1.0, None)
    y = x.clone()
    y[1, 3, 4] = float("nan")
    for _ in range(5):
        got = d2p_amd.soft_sw_affine_with_grads(y, -2.0, -0.5, 1.0, None)
        torch.cuda.empty_cache()
        keep = [i for i in range(B) if i != 1]
        for a, b in zip(want, got):
            assert torch.equal(a[keep], b[keep])


@pytest.mark.parametrize("op", ["soft_sw", "soft_nw"])
@pytest.mark.parametrize("T", [0.2, 1.0])
@pytest.mark.parametrize("B,L1,L2", [(4, 100, 120),     # both sweeps in one launch
                                     (4, 257, 130),     # two parts
                                     (300, 100, 45)])   # one reverse wave a stripe
def test_strong_scores(cuda, B, L1, L2, T, op):
    # one cell each whose factor lies at the upper end of the 32-bit range, 2^121 to 2^127
    # (whose rounding, 2^-24 of 127 bits, adds to that of the ordinary ones on its path)
    s, _ = _inputs(B, L1, L2, False)
    tol = math.hypot(_tol(s, min(L1, L2), T), 8.0 * 2.0 ** -24 * 127.0)
    for b, x in enumerate((84.0, 86.0, 88.0)):
        s[b, L1 // 2, L2 // 2] = x * T
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), -1.0, T, None)
    want = getattr(O.get("oracle64"), op)(s[:4].astype(np.float64), -1.0, T, None)
    _check([x[:4] for x in got], want, s[:4], (-1.0,), T, tol, op == "soft_nw")


@pytest.mark.parametrize("L2", range(189, 206))
@pytest.mark.parametrize("op,gaps", [("soft_nw", (-2.5,)), ("soft_nw_affine", (-3.0, -2.5))])
def test_values_far_below_their_chunk(cuda, op, gaps, L2):
    # the element ends on a run of gaps, 14 bits each: its value lies up to 16 of them below the
    # exponent that its chunk began with, through the end of the 32-bit range
    s, _ = _inputs(2, 100, L2, False)
    s[:, :, 100:] -= 20.0
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), *gaps, 0.25, None)
    want = getattr(O.get("oracle64"), op)(s.astype(np.float64), *gaps, 0.25, None)
    _check(got, want, s, gaps, 0.25, _tol(s, 100, 0.25), True)


def _segments(L1, L2, T, match, penalty):
    """Matches along the diagonal, everything else and the diagonal's middle cell at the
    penalty: (local alignment, affine gaps) one path has both halves, through that cell."""
    s = np.full((L1, L2), penalty, np.float32)
    for i in range(min(L1, L2)):
        s[i, i] = match
    s[min(L1, L2) // 2, min(L1, L2) // 2] = penalty
    return s


@pytest.mark.parametrize("L1,L2", [(60, 60), (60, 250), (300, 310)])
@pytest.mark.parametrize("T,match,penalty,gaps", [
    (1.0, 5.0, -80.0, (-11.0, -1.0)),       # factors within the 32-bit range
    (1.0, 5.0, -90.0, (-11.0, -1.0)),       # below it
    (1.0, 5.0, -110.0, (-11.0, -1.0)),
    (0.5, 5.0, -75.0, (-11.0, -1.0)),
    (0.2, 5.0, -22.0, (-3.0, -0.5)),
    (0.25, 4.0, -100.0, (-3.0, -0.5)),
    (0.2, 9.0, -200.0, (-3.0, -0.5)),       # below the 64-bit range
])
@pytest.mark.parametrize("op", ["soft_sw_affine", "soft_nw_affine"])
def test_mismatches_that_have_to_be_crossed(cuda, op, T, match, penalty, gaps, L1, L2):
    # (local affine alignment has no step from one kind of gap to the other)
    s, _ = _inputs(3, L1, L2, False)
    s[0] = _segments(L1, L2, T, match, penalty)
    s[1, L1 // 2, L2 // 3] = penalty        # a cell that no path has to cross
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), *gaps, T, None)
    want = getattr(O.get("oracle64"), op)(s.astype(np.float64), *gaps, T, None)
    # alpha's rounding, for the elements that the log-domain sweeps take: half an ulp of
    # the value's size in each of the path's cells, to either side
    m = min(L1, L2)
    tol = _tol(s, m, T) + 8.0 * math.sqrt(L1 + L2) * 2.0 ** -24 * float(want[0].max()) / T
    _check(got, want, s, gaps, T, tol, op == "soft_nw_affine")


def _blocks(B, L1, L2, match, masked):
    """Two blocks, with matches along their diagonals, one more in the second; everything outside
    of them masked, three rows and columns between them included."""
    s, _ = _inputs(B, L1, L2, False)
    c1, c2 = int(0.45 * L1), int(0.45 * L2)
    n = min(c1, c2) - 3
    for i in range(n):
        s[:, i, i] = match
    for i in range(n + 1):
        s[:, c1 + i, c2 + i] = match
    s[:, :c1, c2 - 3:] = masked
    s[:, c1 - 3:, :c2] = masked
    return s


@pytest.mark.parametrize("T,match", [(1.0, 2.0), (1.0, 8.0), (0.2, 5.0)])
@pytest.mark.parametrize("masked", [-1e3, -1e9, -1e30])
@pytest.mark.parametrize("op,gaps", [("soft_sw", (-1.0,)), ("soft_nw", (-1.0,)),
                                     ("soft_sw_affine", (-3.0, -0.5)),
                                     ("soft_nw_affine", (-3.0, -0.5))])
@pytest.mark.parametrize("B,L1,L2", [(2, 190, 160), (300, 190, 160)])
def test_masked_blocks(cuda, B, L1, L2, op, gaps, masked, T, match):
    # (local affine alignment: no path has both blocks, and the second one's rows start anew
    # beside gaps that leave the first one, of weights beyond the 64-bit range above 1)
    s = _blocks(B, L1, L2, match, masked)
    got = getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), *gaps, T, None)
    want = getattr(O.get("oracle64"), op)(s[:2].astype(np.float64), *gaps, T, None)
    live = np.where(s[:2] > -100, s[:2], 0)
    tol = _tol(live, min(L1, L2), T) + 8.0 * math.sqrt(L1 + L2) * 2.0 ** -24 * float(
        np.abs(want[0]).max()) / T
    _check([x[:2] for x in got], want, s[:2], gaps, T, tol, "nw" in op)


@pytest.mark.parametrize("op,gaps", [("soft_sw", (-1.0,)), ("soft_nw", (-1.0,)),
                                     ("soft_sw_affine", (-2.0, -0.5)),
                                     ("soft_nw_affine", (-2.0, -0.5))])
@pytest.mark.parametrize("B,L1,L2", [(3, 130, 70), (300, 130, 70), (3, 300, 83)])
def test_infinite_masks_keep_the_sweeps(cuda, B, L1, L2, op, gaps):
    # the factor of -inf and of -1e30 is 0 alike: the same bits, from the same sweeps
    out = []
    for masked in (-1e30, -math.inf):
        s, _ = _inputs(B, L1, L2, False)
        s[:, :, 50:60] = masked
        s[1, 20:, :] = masked
        out.append(getattr(d2p_amd, op + "_with_grads")(torch.from_numpy(s).to(cuda), *gaps, 1.0,
                                                        None))
    for n, (a, b) in enumerate(zip(*out)):
        assert torch.equal(a, b), (n, float((a - b).abs().max()))
