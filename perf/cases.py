"""The calls whose speed this framework is measured by.

A case is one use of a case module's public entry points (``candidate`` with
autograd for a training step, ``forward_only`` for inference) at one size.
``listed()`` names twelve of them, ``draw(rng)`` gives more from the same
ranges, ``prepare`` makes what a program holds before the call, ``run`` is one
pass, ``exact`` the same outputs in 64 bits from plain torch operators.

A training step returns the forward's output and every gradient.
"""

import math
import os
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(REPO, "nl2cuda-kernel-agent_amd")
if PACKAGE not in sys.path:
    sys.path.insert(1, PACKAGE)

DEVICE = "cuda:0"
GAMMA = 0.5           # RBF width of the acceptance workload, rows scaled to unit length
COS_EPS = 1e-8
NORM_EPS = 1e-5       # layernorm
L2N_EPS = 1e-6
MAX_ROW = 4096        # longest row of the power-law matrices


def listed():
    return [
        # Kernel matrix of a small batch: launches and latency count.
        {"name": "rbf_256", "op": "rbf", "n": 256, "m": 256, "d": 64, "mode": "train"},
        # The headline workload: 4096 points against 4096, 64 features.
        {"name": "rbf_4096", "op": "rbf", "n": 4096, "m": 4096, "d": 64, "mode": "train"},
        # Points and features in numbers that are no multiples of a tile.
        {"name": "rbf_3000x2500_d100", "op": "rbf", "n": 3000, "m": 2500, "d": 100,
         "mode": "train"},
        # Embeddings of 128 features compared in pairs (contrastive training).
        {"name": "cosine_2048x4096_d128", "op": "cosine_sim", "n": 2048, "m": 4096, "d": 128,
         "mode": "train"},
        # The acceptance layernorm: 8192 tokens of width 4096.
        {"name": "layernorm_8192x4096", "op": "layernorm", "b": 8192, "d": 4096, "mode": "train"},
        # Row normalisation of an odd width: rows start off any vector boundary.
        {"name": "l2norm_5001x1001", "op": "l2norm_scale", "b": 5001, "d": 1001, "mode": "train"},
        # The reference's default scan, both directions.
        {"name": "scan_4096x4096", "op": "scan", "b": 4096, "d": 4096, "dtype": "float32",
         "mode": "train"},
        # Offsets from counts: few long rows of int32, exact int64 sums, no gradient.
        {"name": "scan_int_64x65536", "op": "scan", "b": 64, "d": 65536, "dtype": "int32",
         "mode": "forward"},
        # A language-model head with an odd vocabulary.
        {"name": "softmax_ce_4096x50257", "op": "softmax_ce", "b": 4096, "c": 50257,
         "mode": "train"},
        # The acceptance SpMV: 2^20 rows of power-law lengths, mean 16.
        {"name": "spmv_zipf_2p20", "op": "spmv", "m": 1 << 20, "k": 1 << 20, "d": 1, "mean": 16,
         "rows": "zipf", "index": "int32", "mode": "train"},
        # The reference's default SpMM: 64 nonzeros in each row, int64 indices.
        {"name": "spmm_4096_d64", "op": "spmv", "m": 4096, "k": 4096, "d": 64, "mean": 64,
         "rows": "uniform", "index": "int64", "mode": "train"},
        # Feature propagation over a graph: many nodes, 32 features, power-law degrees.
        {"name": "spmm_graph_100k_d32", "op": "spmv", "m": 100000, "k": 100000, "d": 32,
         "mean": 16, "rows": "zipf", "index": "int64", "mode": "train"},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["rbf", "cosine_sim", "layernorm", "l2norm_scale", "scan", "softmax_ce",
                     "spmv"])
    mode = rng.choice(["train", "train", "forward"])
    if op in ("rbf", "cosine_sim"):
        # up to the 8192 x 8192 points or 256 features of the tests and benchmark
        while True:
            n, m = _log(rng, 64, 8192), _log(rng, 64, 8192)
            d = rng.choice([64, _log(rng, 4, 256)])
            if n * m * d <= 1 << 31:
                return {"op": op, "n": n, "m": m, "d": d, "mode": mode}
    if op in ("layernorm", "l2norm_scale"):
        while True:
            b, d = _log(rng, 16, 16384), _log(rng, 64, 16384)
            if rng.random() < 0.5:
                d = max(64, d // 64 * 64)
            if b * d <= 1 << 26:
                return {"op": op, "b": b, "d": d, "mode": mode}
    if op == "scan":
        dtype = rng.choice(["float32", "float32", "int32"])
        while True:
            b, d = _log(rng, 1, 16384), _log(rng, 64, 1 << 18)
            if rng.random() < 0.5:
                d = max(64, d // 64 * 64)
            if b * d <= 1 << 25:
                return {"op": op, "b": b, "d": d, "dtype": dtype,
                        "mode": "forward" if dtype == "int32" else mode}
    if op == "softmax_ce":
        while True:
            b, c = _log(rng, 16, 16384), _log(rng, 10, 131072)
            if b * c <= 1 << 27:
                return {"op": op, "b": b, "c": c, "mode": mode}
    while True:
        m, k = _log(rng, 1000, 1 << 20), _log(rng, 1000, 1 << 20)
        d = rng.choice([1, _log(rng, 2, 128)])
        mean = _log(rng, 4, 64)
        if m * mean <= 1 << 24 and m * mean * d <= 1 << 26 and (m + k) * d <= 1 << 25:
            return {"op": op, "m": m, "k": k, "d": d, "mean": mean,
                    "rows": rng.choice(["zipf", "uniform"]),
                    "index": rng.choice(["int32", "int64"]), "mode": mode}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE)


def _row_lengths(case):
    """Row lengths before shuffling: a function of the case alone, so every
    seed has the same number of nonzeros.  "zipf": the quantiles of a power
    law of exponent 1.5 clipped to [1, 4096], rescaled to the mean."""
    m, mean = case["m"], case["mean"]
    if case["rows"] == "uniform":
        return torch.full((m,), mean, dtype=torch.int64, device=DEVICE)
    cap = min(MAX_ROW, case["k"])
    u = (torch.arange(m, dtype=torch.float64, device=DEVICE) + 0.5) / m
    raw = u.pow(-2.0).clamp(max=MAX_ROW)
    lens = (raw * (mean * m / raw.sum())).floor().clamp(1, cap).to(torch.int64)
    # the rounding's remainder, one to each of the first rows that may take it
    short = mean * m - int(lens.sum())
    if short > 0:
        room = (lens < cap).nonzero().flatten()
        each = -(-short // room.numel())
        add = torch.full((room.numel(),), each, dtype=torch.int64, device=DEVICE)
        over = each * room.numel() - short
        if over:
            add[-over:] -= 1
        lens[room] += add
    return lens


def _nnz(case):
    return int(_row_lengths(case).sum())


def _csr(case, g):
    lens = _row_lengths(case)
    lens = lens[torch.randperm(case["m"], generator=g, device=DEVICE)]
    row_ptr = torch.zeros(case["m"] + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(lens, 0, out=row_ptr[1:])
    rows = torch.repeat_interleave(torch.arange(case["m"], device=DEVICE), lens)
    cols = torch.randint(0, case["k"], (rows.numel(),), generator=g, device=DEVICE)
    cols = torch.sort(rows * case["k"] + cols).values - rows * case["k"]  # ascending in a row
    dtype = getattr(torch, case["index"])
    return row_ptr.to(dtype), cols.to(dtype)


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    train = case["mode"] == "train"
    state = {"op": op, "train": train, "params": {}}
    if op == "rbf":
        s = 1.0 / math.sqrt(case["d"])
        inputs = {"X": _randn(g, case["n"], case["d"]) * s,
                  "Y": _randn(g, case["m"], case["d"]) * s}
        leaves, out = ["X", "Y"], (case["n"], case["m"])
        state["params"] = {"gamma": GAMMA}
    elif op == "cosine_sim":
        inputs = {"A": _randn(g, case["n"], case["d"]), "B": _randn(g, case["m"], case["d"])}
        leaves, out = ["A", "B"], (case["n"], case["m"])
        state["params"] = {"eps": COS_EPS}
    elif op == "layernorm":
        inputs = {"X": _randn(g, case["b"], case["d"]),
                  "gamma": 1.0 + 0.1 * _randn(g, case["d"]), "beta": 0.1 * _randn(g, case["d"])}
        leaves, out = ["X", "gamma", "beta"], (case["b"], case["d"])
        state["params"] = {"eps": NORM_EPS}
    elif op == "l2norm_scale":
        inputs = {"X": _randn(g, case["b"], case["d"]), "g": _randn(g, case["d"])}
        leaves, out = ["X", "g"], (case["b"], case["d"])
        state["params"] = {"eps": L2N_EPS}
    elif op == "scan":
        if case["dtype"] == "int32":
            inputs = {"X": torch.randint(-1000, 1001, (case["b"], case["d"]), generator=g,
                                         device=DEVICE, dtype=torch.int32)}
        else:
            inputs = {"X": _randn(g, case["b"], case["d"])}
        leaves, out = ["X"], (case["b"], case["d"])
    elif op == "softmax_ce":
        inputs = {"logits": _randn(g, case["b"], case["c"]) * 2.0,
                  "labels": torch.randint(0, case["c"], (case["b"],), generator=g, device=DEVICE)}
        leaves, out = ["logits"], ()
    else:
        row_ptr, col_idx = _csr(case, g)
        inputs = {"row_ptr": row_ptr, "col_idx": col_idx, "vals": _randn(g, col_idx.numel()),
                  "X": _randn(g, case["k"], case["d"])}
        leaves, out = ["vals", "X"], (case["m"], case["d"])
    state["inputs"] = inputs
    if train:
        # the gradient that comes back from the rest of the model; a loss starts at 1
        state["upstream"] = (torch.ones((), device=DEVICE) if op == "softmax_ce"
                             else _randn(g, *out))
        state["leaves"] = leaves
        for name in leaves:
            inputs[name].requires_grad_(True)
    return state


def _op(name):
    if name == "rbf":
        from cases.rbf import op
    elif name == "cosine_sim":
        from cases.cosine_sim import op
    elif name == "layernorm":
        from cases.layernorm import op
    elif name == "l2norm_scale":
        from cases.l2norm_scale import op
    elif name == "scan":
        from cases.scan import op
    elif name == "softmax_ce":
        from cases.softmax_ce import op
    else:
        from cases.spmv import op
    return op


def run(state):
    op = _op(state["op"])
    inputs = state["inputs"]
    if not state["train"]:
        return {"out": op.forward_only(inputs, state["params"])}
    out = op.candidate(inputs, state["params"])
    grads = torch.autograd.grad(out, [inputs[k] for k in state["leaves"]], state["upstream"])
    return {"out": out.detach(), **{"d" + k: v for k, v in zip(state["leaves"], grads)}}


# -------------------------------------------------------------------- work
def work(case):
    op, train = case["op"], case["mode"] == "train"
    if op in ("rbf", "cosine_sim"):
        n, m, d = case["n"], case["m"], case["d"]
        nbytes, flops = 4 * n * m + 4 * d * (n + m), 2 * n * m * d
        if train:  # rbf reads dK and the saved K, cosine dS alone
            nbytes += (8 if op == "rbf" else 4) * n * m + 8 * d * (n + m)
            flops += 4 * n * m * d
    elif op in ("layernorm", "l2norm_scale"):
        b, d = case["b"], case["d"]
        nbytes, flops = 8 * b * d + 8 * d, 5 * b * d
        if train:
            nbytes, flops = nbytes + 12 * b * d + 12 * d + 8 * b, flops + 10 * b * d
    elif op == "scan":
        n = case["b"] * case["d"]
        nbytes, flops = (12 if case["dtype"] == "int32" else 8) * n, n
        if train:
            nbytes, flops = 2 * nbytes, 2 * flops
    elif op == "softmax_ce":
        b, c = case["b"], case["c"]
        nbytes, flops = 4 * b * c + 12 * b, 4 * b * c
        if train:
            nbytes, flops = nbytes + 8 * b * c + 12 * b, flops + 4 * b * c
    else:
        m, k, d = case["m"], case["k"], case["d"]
        nnz = case["mean"] * m
        s = 8 if case["index"] == "int64" else 4
        nbytes, flops = nnz * (s + 4) + (m + 1) * s + 4 * d * (k + m), 2 * nnz * d
        if train:
            nbytes += nnz * (s + 8) + (m + 1) * s + 4 * d * (2 * k + m)
            flops += 4 * nnz * d
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["op"] == "scan" and case["dtype"] == "int32":
        return "exact"
    # Measured against 64 bits: at most 3.5e-7 (the pairwise gradients), 1e-7 elsewhere; two
    # orders of the same 32-bit sums differ by as much.
    return {"rel": 2e-6}


# ------------------------------------------------------------------- exact
def _pair_grads(W, X, Y):
    """(rowsum, colsum, W Y, W^T X)."""
    return W.sum(1, keepdim=True), W.sum(0).unsqueeze(1), W @ Y, W.t().contiguous() @ X


def _unit_grad(A, norm, inv, dAh):
    """d/dA of A * inv with inv = 1 / (norm + eps)."""
    dot = (dAh * A).sum(1, keepdim=True)
    return dAh * inv - A * (dot * inv * inv / norm.clamp_min(1e-300))


def exact(case, seed):
    state = prepare(case, seed)
    op, train = state["op"], state["train"]
    x = {k: (v.detach().double() if v.is_floating_point() else v)
         for k, v in state["inputs"].items()}
    up = state["upstream"].double() if train else None
    if op == "rbf":
        X, Y = x["X"], x["Y"]
        d2 = X.square().sum(1, keepdim=True) + Y.square().sum(1) - 2.0 * (X @ Y.t().contiguous())
        K = torch.exp(-GAMMA * d2)
        got = {"out": K}
        if train:
            row, col, WY, WX = _pair_grads(up * K, X, Y)
            got["dX"] = -2.0 * GAMMA * (row * X - WY)
            got["dY"] = -2.0 * GAMMA * (col * Y - WX)
        return got
    if op == "cosine_sim":
        A, B = x["A"], x["B"]
        na, nb = A.norm(dim=1, keepdim=True), B.norm(dim=1, keepdim=True)
        ia, ib = 1.0 / (na + COS_EPS), 1.0 / (nb + COS_EPS)
        got = {"out": (A * ia) @ (B * ib).t().contiguous()}
        if train:
            _, _, SB, SA = _pair_grads(up, A * ia, B * ib)
            got["dA"] = _unit_grad(A, na, ia, SB)
            got["dB"] = _unit_grad(B, nb, ib, SA)
        return got
    if op == "layernorm":
        X, gamma = x["X"], x["gamma"]
        mean = X.mean(1, keepdim=True)
        rstd = ((X - mean).square().mean(1, keepdim=True) + NORM_EPS).rsqrt()
        h = (X - mean) * rstd
        got = {"out": h * gamma + x["beta"]}
        if train:
            dh = up * gamma
            got["dX"] = rstd * (dh - dh.mean(1, keepdim=True)
                                - h * (dh * h).mean(1, keepdim=True))
            got["dgamma"], got["dbeta"] = (up * h).sum(0), up.sum(0)
        return got
    if op == "l2norm_scale":
        X, scale = x["X"], x["g"]
        inv = (X.square().sum(1, keepdim=True) + L2N_EPS).rsqrt()
        h = X * inv
        got = {"out": h * scale}
        if train:
            dh = up * scale
            got["dX"] = inv * (dh - h * (dh * h).sum(1, keepdim=True))
            got["dg"] = (up * h).sum(0)
        return got
    if op == "scan":
        got = {"out": torch.cumsum(x["X"], 1)}
        if train:
            got["dX"] = torch.cumsum(up.flip(1), 1).flip(1)
        return got
    if op == "softmax_ce":
        logits, labels = x["logits"], x["labels"]
        lse = torch.logsumexp(logits, 1, keepdim=True)
        got = {"out": (lse - logits.gather(1, labels.unsqueeze(1))).mean()}
        if train:
            p = torch.exp(logits - lse)
            p.scatter_add_(1, labels.unsqueeze(1),
                           torch.full((labels.numel(), 1), -1.0, dtype=p.dtype, device=DEVICE))
            got["dlogits"] = p * (up / labels.numel())
        return got
    row_ptr, cols, vals, X = x["row_ptr"].long(), x["col_idx"].long(), x["vals"], x["X"]
    rows = torch.repeat_interleave(torch.arange(case["m"], device=DEVICE),
                                   row_ptr[1:] - row_ptr[:-1])
    out = torch.zeros(case["m"], case["d"], dtype=torch.float64, device=DEVICE)
    got = {"out": out.index_add_(0, rows, vals.unsqueeze(1) * X[cols])}
    if train:
        dY = up[rows]
        got["dvals"] = (dY * X[cols]).sum(1)
        got["dX"] = torch.zeros_like(X).index_add_(0, cols, vals.unsqueeze(1) * dY)
    return got
