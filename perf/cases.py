"""The work that users have d2p_amd do, as timed cases: soft alignment forward and
backward through the public functions, over the sizes of the repository's own tests and
benchmark configurations, with ragged and odd shapes beside the round ones.

Every case runs the public entry point of its family once: ``value`` cases the forward
and the gradient of the summed (or averaged) alignment value, ``marginal`` cases the
gradient of a loss on the alignment matrix itself (the second-order path), ``hvp`` cases
the explicit Hessian-vector product.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import d2p_amd


def listed():
    return [
        # the smallest call in use: two short sequences (unit tests, notebooks, per-pair
        # scoring), where launches and the dependency chain of one table are everything
        dict(name="sw_pair", op="sw", mode="value", B=2, L1=100, L2=120, T=1.0, scale=1.0,
             ragged=False, learn=False),
        # the benchmark's headline: a training batch of protein-length pairs
        dict(name="sw_batch", op="sw", mode="value", B=256, L1=512, L2=512, T=1.0, scale=1.0,
             ragged=False, learn=False),
        # a padded batch of unequal sequences with a learnable gap and temperature
        dict(name="sw_learn_ragged", op="sw", mode="value", B=48, L1=300, L2=411, T=0.7,
             scale=1.5, ragged=True, learn=True),
        # genome-scale rows: few, long elements
        dict(name="sw_long", op="sw", mode="value", B=16, L1=4096, L2=4096, T=1.0, scale=1.0,
             ragged=False, learn=False),
        # a loss on the alignment matrix: its gradient runs the second-order sweeps
        dict(name="sw_marginal_loss", op="sw", mode="marginal", B=64, L1=384, L2=384, T=1.0,
             scale=1.0, ragged=False, learn=False),
        # curvature products on long elements
        dict(name="sw_hvp_long", op="sw", mode="hvp", B=16, L1=4096, L2=4096, T=1.0, scale=1.0,
             ragged=False, learn=False),
        # affine gaps with substitution-matrix-like penalties on a ragged batch
        dict(name="affine_ragged", op="affine", mode="value", B=64, L1=1024, L2=1024, T=0.5,
             scale=2.0, ragged=True, learn=False),
        # global alignment of odd-sized pairs
        dict(name="nw_odd", op="nw", mode="value", B=96, L1=301, L2=277, T=1.0, scale=1.0,
             ragged=False, learn=False),
        dict(name="nw_affine", op="nw_affine", mode="value", B=32, L1=500, L2=450, T=1.0,
             scale=1.0, ragged=True, learn=False),
        # time series under a given cost matrix (squared distances of 64-d features)
        dict(name="dtw_batch", op="dtw", mode="value", B=512, L1=256, L2=256, T=0.1, scale=1.0,
             ragged=False, learn=False, band=0, D=64),
        # long time series under a Sakoe-Chiba band
        dict(name="dtw_band_long", op="dtw", mode="value", B=16, L1=4096, L2=4096, T=1.0,
             scale=1.0, ragged=False, learn=False, band=64, D=0),
        # time series from their features, with gradients into the features
        dict(name="dtw_features", op="dtw_features", mode="value", B=512, L1=256, L2=256, T=0.1,
             scale=1.0, ragged=False, learn=False, band=0, D=64),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sw", "sw", "sw", "affine", "affine", "nw", "nw_affine", "dtw", "dtw",
                     "dtw_features"])
    L1, L2 = _log_uniform(rng, 24, 2048), _log_uniform(rng, 24, 2048)
    if rng.random() < 0.5:                  # pairs of like length, as most are
        L2 = max(24, min(2048, int(L1 * rng.uniform(0.8, 1.25))))
    most = min(512, max(1, (1 << 25) // (L1 * L2)))
    case = dict(op=op, mode="value", B=_log_uniform(rng, 1, most), L1=L1, L2=L2,
                T=rng.choice([0.5, 0.7, 1.0, 1.0, 2.0]), scale=rng.choice([1.0, 1.0, 2.0]),
                ragged=rng.random() < 0.4, learn=False)
    if op == "sw":
        case["mode"] = rng.choice(["value", "value", "marginal", "hvp"])
        case["learn"] = case["mode"] == "value" and rng.random() < 0.5
    if op in ("affine", "nw", "nw_affine") and rng.random() < 0.25:
        case["mode"] = "marginal"
    if op in ("dtw", "dtw_features"):
        case["T"] = rng.choice([0.1, 0.5, 1.0])
        case["band"] = rng.choice([0, 0, 16, 64]) if op == "dtw" else 0
        if case["band"] and abs(L1 - L2) > 16:
            case["band"] = 0
        case["D"] = rng.choice([8, 33, 64]) if op == "dtw_features" else rng.choice([0, 64])
    return case


GAP = -1.0
AFFINE = (-11.0, -1.0)       # substitution-matrix-like penalties
NW_AFFINE = (-2.0, -0.5)     # the functions' defaults


def _tensors(case, seed, device):
    """The case's inputs, from the seed alone."""
    g = torch.Generator(device=device).manual_seed(seed)
    B, L1, L2 = case["B"], case["L1"], case["L2"]

    def randn(*shape):
        return torch.randn(shape, generator=g, device=device)

    x = {}
    if case["op"] == "dtw_features":
        x["x"], x["y"] = randn(B, L1, case["D"]), randn(B, L2, case["D"])
    elif case["op"] == "dtw":
        if case["D"]:
            a, b = randn(B, L1, case["D"]), randn(B, L2, case["D"])
            x["m"] = (a.square().sum(-1)[:, :, None] + b.square().sum(-1)[:, None, :]
                      - 2 * torch.bmm(a, b.transpose(1, 2).contiguous())).clamp_(min=0)
        else:
            x["m"] = randn(B, L1, L2).abs_() * case["scale"]
    else:
        x["m"] = randn(B, L1, L2) * case["scale"]
    if case["mode"] in ("hvp", "marginal"):
        x["v"] = randn(B, L1, L2)
    if case["ragged"]:
        r = torch.rand((B, 2), generator=g, device=device)
        most = torch.tensor([L1, L2], device=device)
        low = torch.clamp(most // 4, min=1)
        x["lengths"] = (low + (r * (most - low + 1)).floor().long()).clamp(max=most).int()
    return x


def prepare(case, seed):
    dev = torch.device("cuda")
    x = _tensors(case, seed, dev)
    state = dict(case=dict(case), lengths=x.get("lengths"), v=x.get("v"))
    state["leaves"] = [x[k].requires_grad_(case["mode"] != "hvp") for k in ("x", "y", "m")
                       if k in x]
    if case["learn"]:
        state["gap"] = torch.tensor([GAP], device=dev, requires_grad=True)
        state["T"] = torch.tensor([case["T"]], device=dev, requires_grad=True)
    return state


def run(state):
    c, lengths, leaves = state["case"], state["lengths"], state["leaves"]
    op, T, m = c["op"], c["T"], state["leaves"][0]
    if c["mode"] == "hvp":
        return {"hvp": d2p_amd.soft_sw_hvp(m, state["v"], GAP, T, lengths)}
    params = []
    if op == "sw":
        if c["learn"]:
            params = [state["gap"], state["T"]]
            res = d2p_amd.soft_sw(m, params[0], params[1], lengths)
        else:
            res = d2p_amd.soft_sw(m, GAP, T, lengths)
    elif op == "affine":
        res = d2p_amd.soft_sw_affine(m, AFFINE[0], AFFINE[1], T, lengths)
    elif op == "nw":
        res = d2p_amd.soft_nw(m, GAP, T, lengths)
    elif op == "nw_affine":
        res = d2p_amd.soft_nw_affine(m, NW_AFFINE[0], NW_AFFINE[1], T, lengths)
    elif op == "dtw":
        res = d2p_amd.soft_dtw(m, T, c["band"], lengths)
    else:
        res = d2p_amd.soft_dtw_sqeuclidean(leaves[0], leaves[1], T, c["band"], lengths)
    value, align = res[0], res[1]
    if c["mode"] == "marginal":
        loss = (align * state["v"]).sum()
    else:
        loss = value.mean() if c["learn"] else value.sum()
    grads = torch.autograd.grad(loss, leaves + params)
    return {"value": value.detach(), "align": align.detach(), "grads": list(grads)}


def work(case):
    cells = case["B"] * case["L1"] * case["L2"]
    feats = case["B"] * (case["L1"] + case["L2"]) * case.get("D", 0)
    if case["op"] == "dtw_features":
        # features in and their gradients out, the alignment out; the distance product
        # and the two gradient products
        return {"bytes": 4 * (2 * feats + cells), "flops": 6.0 * cells * case["D"]}
    # matrix in, alignment out, gradient out; a direction or loss weight in
    n = {"value": 3, "marginal": 4, "hvp": 3}[case["mode"]]
    # per cell: one exponential and the handful of products and sums of each direction
    per = {"sw": 12, "nw": 12, "dtw": 10, "affine": 30, "nw_affine": 36}[case["op"]]
    return {"bytes": 4.0 * n * cells, "flops": per * cells * (1 if case["mode"] == "value" else 2)}


def tolerance(case):
    # four times what was seen against the 64-bit values.  float32 tables hold values that
    # grow with the length of the paths, and the exponentials turn their rounding into a
    # relative error of the marginals; second derivatives and low temperatures amplify
    # it.  Costs of 2 D per cell on average make the largest values.
    if case.get("D", 0):
        rel = 5e-3
    else:
        rel = 1.6e-4 * max(0.25, (case["L1"] + case["L2"]) / 1024.0)
        rel *= 2 if case["op"] == "dtw" else 1
        if case["mode"] != "value":
            rel *= 8 / min(1.0, case["T"])
    return {"rel": min(rel, 2e-2), "max": min(60 * rel, 0.8)}


# ------------------------------------------------------------------ exact values

NEG = -1e30


def _diagonals(m, fill=0.0):
    """[B, L1, L2] as the list of its anti-diagonals, each [B, L1] indexed by the row."""
    B, L1, L2 = m.shape
    W = L1 + L2 - 1
    x = F.pad(m, (0, W + 1 - L2), value=fill).reshape(B, -1)[:, :L1 * W]
    return x.reshape(B, L1, W).permute(2, 0, 1).contiguous().unbind(0)


def _lse(*terms):
    return torch.logsumexp(torch.stack(terms), 0)


def _down(v, first):
    """Row i of the result is row i - 1 of v; row 0 is `first`."""
    B = v.shape[0]
    f = first if isinstance(first, torch.Tensor) else torch.tensor(float(first))
    f = f.to(v).reshape(1, 1).expand(B, 1)
    return torch.cat([f, v[:, :-1]], 1)


def _value(op, m, params, lengths, band):
    """The alignment value [B] in 64 bits, differentiable, by anti-diagonals."""
    T = params[-1]
    B, L1, L2 = m.shape
    dev = m.device
    rows = torch.arange(L1, device=dev)
    diags = _diagonals(m)
    none = torch.full((B, L1), NEG, dtype=m.dtype, device=dev)
    b = torch.arange(B, device=dev)
    l1, l2 = lengths[:, 0].long(), lengths[:, 1].long()
    ends = [[], [], []]
    n_states = 3 if op in ("affine", "nw_affine") else 1
    if op in ("sw", "nw"):
        gap = params[0] / T
        col0 = ((rows + 1) * gap).expand(B, L1) if op == "nw" else none
    elif n_states == 3:
        go, ge = params[0] / T, params[1] / T
        col0 = (go + rows * ge).expand(B, L1) if op == "nw_affine" else none
    else:
        col0 = none
    p1 = p2 = [none, col0 if n_states == 3 else none, none] if n_states == 3 else [col0]
    for d, raw in enumerate(diags):
        s = raw / T
        inside = (rows <= d)                    # j = d - i >= 0
        if op == "sw":
            up, left, diag = _down(p1[0], NEG), p1[0], _down(p2[0], NEG)
            new = [_lse(diag + s, s, up + gap, left + gap)]
            edge = [none]
        elif op == "nw":
            up, left, diag = _down(p1[0], (d + 1) * gap), p1[0], _down(p2[0], d * gap)
            new = [_lse(diag + s, up + gap, left + gap)]
            edge = [col0]
        elif op == "dtw":
            up, left, diag = _down(p1[0], NEG), p1[0], _down(p2[0], 0.0 if d == 0 else NEG)
            x = _lse(diag, up, left) - s
            if band > 0:
                i, j = (rows + 1).float(), (d - rows + 1).float()
                e = (i * l2[:, None].float()) / l1[:, None].float()
                x = torch.where((j - e).abs() <= band, x, none)
            new, edge = [torch.clamp(x, min=NEG)], [none]
        elif op == "affine":
            dg = [_down(v, NEG) for v in p2]
            up = [_down(v, NEG) for v in p1]
            new = [_lse(dg[0] + s, dg[1] + s, dg[2] + s, s), _lse(up[0] + go, up[1] + ge),
                   _lse(p1[0] + go, p1[2] + ge)]
            edge = [none, none, none]
        else:
            top = go + (d - 1) * ge             # the D state of row 0, column d
            dg = [_down(p2[0], 0.0 if d == 0 else NEG), _down(p2[1], NEG),
                  _down(p2[2], NEG if d == 0 else top)]
            up = [_down(p1[0], NEG), _down(p1[1], NEG), _down(p1[2], top + ge)]
            new = [_lse(*dg) + s, _lse(up[0] + go, up[1] + ge, up[2] + go),
                   _lse(p1[0] + go, p1[1] + go, p1[2] + ge)]
            edge = [none, col0, none]
        new = [torch.where(inside, v, e) for v, e in zip(new, edge)]
        for k, v in enumerate(new):
            ends[k].append(v)
        p2, p1 = p1, new
    tables = [torch.stack(e) for e in ends[:n_states]]          # [W, B, L1]
    if op in ("sw", "affine"):
        j = torch.arange(L1 + L2 - 1, device=dev)[:, None] - rows   # [W, L1]
        valid = ((j[:, None] >= 0) & (j[:, None] < l2[None, :, None])
                 & (rows < l1[:, None])[None])
        tot = [torch.zeros(B, dtype=m.dtype, device=dev)]
        for t in tables:
            t = torch.where(valid, t, torch.full_like(t, NEG))
            tot.append(torch.logsumexp(torch.logsumexp(t, 2), 0))
        return T * _lse(*tot)
    last = [t[l1 + l2 - 2, b, l1 - 1] for t in tables]
    if op == "nw_affine":
        return T * _lse(*last)
    return (-T if op == "dtw" else T) * last[0]


def exact(case, seed):
    cells = case["L1"] * case["L2"]
    if case["mode"] != "value" and case["B"] * cells > 24e6:
        return None                             # the double backward's tables
    dev = torch.device("cuda")
    x = {k: v.double() if v.is_floating_point() else v
         for k, v in _tensors(case, seed, dev).items()}
    lengths = x.get("lengths")
    if lengths is None:
        lengths = torch.tensor([[case["L1"], case["L2"]]] * case["B"], device=dev)
    op = case["op"]
    pars = {"sw": (GAP,), "nw": (GAP,), "affine": AFFINE, "nw_affine": NW_AFFINE}.get(op, ())
    params = [torch.tensor(float(torch.tensor(p)), dtype=torch.float64, device=dev,
                           requires_grad=True) for p in pars + (case["T"],)]
    if op == "dtw_features":
        leaves = [x["x"].requires_grad_(), x["y"].requires_grad_()]
        m = (leaves[0].square().sum(-1)[:, :, None] + leaves[1].square().sum(-1)[:, None, :]
             - 2 * torch.bmm(leaves[0], leaves[1].transpose(1, 2).contiguous()))
        mm = m.detach().requires_grad_()
    else:
        mm = x["m"].requires_grad_()
        leaves = [mm]
    second = case["mode"] != "value"
    value = _value("dtw" if op == "dtw_features" else op, mm, params, lengths,
                   case.get("band", 0))
    wanted = [mm] + params
    first = torch.autograd.grad(value.sum(), wanted, create_graph=second, allow_unused=True)
    if case["mode"] == "hvp":
        return {"hvp": torch.autograd.grad((first[0] * x["v"]).sum(), mm)[0]}
    align = first[0]
    if second:
        grads = [torch.autograd.grad((align * x["v"]).sum(), mm)[0]]
    elif op == "dtw_features":
        grads = list(torch.autograd.grad(m, leaves, align))
    elif case["learn"]:
        grads = [align / case["B"]] + [g.reshape(1) / case["B"] for g in first[1:]]
    else:
        grads = [align]
    return {"value": value.detach(), "align": align.detach(), "grads": grads}
