"""SpMM where a row or column crosses the edges of its kernels: the backward's
column buckets (more than 16384 columns: bucket and part edges, columns that
hold most of the entries, widths with a ragged last lane) and the forward's
rows shared by a workgroup (more than 64 entries per lane group).  Against
float64, at a 2-norm error of 2^-24 sqrt(n) / sqrt(3) of the result (n
roundings of a sum of n independent terms), n the longest row or column, and
three roundings more."""

import math

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _csr(lens, k, seed, hub):
    g = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    col = g.integers(0, k, ptr[-1])
    if hub:  # half of the entries in three columns, one of them the last
        at = g.random(ptr[-1]) < 0.5
        col[at] = g.choice([0, 777, k - 1], int(at.sum()))
    return torch.from_numpy(ptr), torch.from_numpy(col)


def _check(lens, k, d, idx, hub=False, seed=0):
    from cases.spmv import op
    announce(f"spmm buckets rows={len(lens)} K={k} D={d} {idx} hub={hub}")
    ptr, col = _csr(np.asarray(lens), k, seed, hub)
    m, nnz = len(lens), col.numel()
    g = torch.Generator().manual_seed(seed)
    vals, X, G = (torch.randn(*s, generator=g) for s in ((nnz,), (k, d), (m, d)))
    v, x = vals.cuda().requires_grad_(True), X.cuda().requires_grad_(True)
    Y = op.candidate({"row_ptr": ptr.to(idx).cuda(), "col_idx": col.to(idx).cuda(), "vals": v,
                      "X": x}, {})
    dv, dx = torch.autograd.grad(Y, [v, x], G.cuda())
    torch.cuda.synchronize()
    rows = torch.repeat_interleave(torch.arange(m), ptr[1:] - ptr[:-1])
    vd, Xd, Gd = vals.double(), X.double(), G.double()
    want = {"Y": (Y, torch.zeros(m, d, dtype=torch.float64).index_add_(
                      0, rows, vd[:, None] * Xd[col]), int(max(lens))),
            "dvals": (dv, (Gd[rows] * Xd[col]).sum(1), d),
            "dX": (dx, torch.zeros(k, d, dtype=torch.float64).index_add_(
                      0, col, vd[:, None] * Gd[rows]), int(torch.bincount(col).max()))}
    for name, (got, ref, n) in want.items():
        tol = 2.0 ** -24 * (3 + math.sqrt(n / 3))
        err = float((got.detach().cpu().double() - ref).norm() / ref.norm())
        print(f"  {name}: {err:.2e} of {tol:.2e}")
        assert err <= tol, name


@pytest.mark.parametrize("d", [2, 3, 4, 5, 7, 32, 33, 64, 127, 130, 256, 300])
@pytest.mark.parametrize("k", [16385, 40001])
def test_spmm_column_buckets(k, d):
    lens = np.random.default_rng(d).integers(0, 30, 700)
    _check(lens, k, d, torch.int64 if d % 2 else torch.int32, seed=d)


@pytest.mark.parametrize("d", [4, 33])
@pytest.mark.parametrize("m,mean", [(3000, 20), (9000, 70)])
def test_spmm_hub_columns(m, mean, d):
    """Buckets of several parts (over 8192 entries, added with atomics) and
    columns that cross from one lane group to the next; 9000 x 70 entries
    take the larger scatter tiles."""
    lens = np.full(m, mean)
    _check(lens, 20000, d, torch.int32, hub=True, seed=m)


@pytest.mark.parametrize("m,mean,k,d", [(1 << 18, 64, 20000, 2), (1 << 20, 15, 1 << 20, 3)])
def test_spmm_many_entries(m, mean, k, d):
    """More entries than 8192 buckets hold in one round of the gather each."""
    from cases.spmv import op
    lib = op._lib()
    assert lib.spmv_backward_best_workspace_bytes(m, k, d, m * mean) >= 16 * m * mean
    _check(np.full(m, mean), k, d, torch.int32, seed=d)


@pytest.mark.parametrize("d", [1 + 1, 6, 16, 20, 40, 100, 260])
def test_spmm_long_rows(d):
    """Rows one short of, at and past the length a workgroup shares, between
    empty and single-entry ones."""
    lens = [0, 1, 63, 64, 65, 127, 128, 129, 255, 257, 1, 0, 513, 1025, 2, 3000, 0, 1] * 3 + [4000]
    _check(lens, 500, d, torch.int64, seed=d)


def test_spmm_bucket_route_needs_its_workspace():
    """A caller with the smaller workspace (none, past 16384 columns) still
    gets dX, through atomics."""
    from cases.spmv import op
    from framework import capi
    m, k, d = 900, 20000, 8
    announce("spmm without the bucket workspace")
    lib = op._lib()
    ptr, col = _csr(np.full(m, 11), k, 1, False)
    nnz = col.numel()
    assert lib.spmv_backward_workspace_bytes(m, k, d, nnz) == 0
    assert lib.spmv_backward_best_workspace_bytes(m, k, d, nnz) >= 16 * nnz
    ptr, col = ptr.int().cuda(), col.int().cuda()
    vals, X, G = torch.randn(nnz).cuda(), torch.randn(k, d).cuda(), torch.randn(m, d).cuda()
    dv0, dx0 = op.spmv_backward(ptr, col, vals, X, G)
    dv, dx = torch.empty_like(vals), torch.empty_like(X)
    P = capi.ptr
    st = lib.spmv_backward_f32_i32(P(ptr), P(col), P(vals), P(X), P(G), P(dv), P(dx), m, k, d, nnz,
                                   None, 0, capi.stream_of(X))
    capi.check(st, lib.spmv_last_error, "spmv_backward")
    torch.cuda.synchronize()
    assert float((dx - dx0).norm() / dx0.norm()) < 1e-6
    assert float((dv - dv0).norm() / dv0.norm()) < 1e-6


@pytest.mark.parametrize("d", [3, 7, 8, 13, 16, 33, 60, 64, 128])
@pytest.mark.parametrize("k", [1, 5, 20, 40, 80])
def test_spmm_few_long_columns(k, d):
    """Few columns of many entries: 1 to 16 lane groups share a column."""
    lens = np.random.default_rng(k).integers(0, 30, 700)
    _check(lens, k, d, torch.int64 if d % 2 else torch.int32, seed=d)


@pytest.mark.parametrize("d", [3, 4, 5, 6, 7, 33, 130])
def test_spmm_bucket_infinities(d):
    """An infinite entry of X, dY or vals reaches the outputs it belongs to and
    no other: lanes that share a row's last four columns keep apart."""
    from cases.spmv import op
    announce(f"spmm buckets with infinities, D={d}")
    m, k = 700, 20000
    ptr, col = _csr(np.full(m, 9), k, d, False)
    g = torch.Generator().manual_seed(d)
    vals, X, G = (torch.randn(*s, generator=g) for s in ((9 * m,), (k, d), (m, d)))
    # column d - 4 is loaded by the last lane, and another's where d % 4 != 0
    X[col[5], max(d - 4, 0)], X[col[900], d - 1] = math.inf, -math.inf
    G[300, d - 2] = math.inf
    vals[4000] = math.inf
    dv, dx = op.spmv_backward(ptr.int().cuda(), col.int().cuda(), vals.cuda(), X.cuda(), G.cuda())
    rows = torch.repeat_interleave(torch.arange(m), 9)
    want_v = (G[rows].double() * X[col].double()).sum(1)
    want_x = torch.zeros(k, d, dtype=torch.float64).index_add_(
        0, col, vals.double()[:, None] * G[rows].double())
    for name, got, want in (("dvals", dv.cpu(), want_v), ("dX", dx.cpu(), want_x)):
        assert torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5, equal_nan=True), name


@pytest.mark.parametrize("hub", [False, True])
def test_spmm_bucket_backward_graph_replays_with_new_inputs(hub):
    """The route captured once (counts cleared by a kernel, places reserved with
    atomics) and replayed on new dY, with buckets of one part and of several:
    every replay against float64 and an eager call, whose additions come in
    another order."""
    from test_gpu_graph_capture import _capture
    from cases.spmv import op
    m, k, d = 4000, 20000, 8
    announce(f"spmm buckets graph capture, hub={hub}")
    ptr, col = _csr(np.full(m, 20), k, 3, hub)
    g = torch.Generator().manual_seed(3)
    vals, X = torch.randn(20 * m, generator=g), torch.randn(k, d, generator=g)
    args = [t.cuda() for t in (ptr.int(), col.int(), vals, X)]
    dy = torch.zeros(m, d, device="cuda")
    graph, (dv, dx) = _capture(lambda: op.spmv_backward(*args, dy))
    rows = torch.repeat_interleave(torch.arange(m), 20)
    tol = 2.0 ** -24 * (3 + math.sqrt(int(torch.bincount(col).max()) / 3))
    for seed in range(4):
        G = torch.randn(m, d, generator=g)
        dy.copy_(G.cuda())
        graph.replay()
        torch.cuda.synchronize()
        want = torch.zeros(k, d, dtype=torch.float64).index_add_(
            0, col, vals.double()[:, None] * G[rows].double())
        want_v = (G[rows].double() * X[col].double()).sum(1)
        edv, edx = op.spmv_backward(*args, dy.clone())
        torch.cuda.synchronize()
        for name, a, b in (("dX", dx, want), ("eager dX", edx, want), ("dvals", dv, want_v)):
            err = float((a.cpu().double() - b).norm() / b.norm())
            print(f"  replay {seed} {name}: {err:.2e} of {tol:.2e}")
            assert err <= tol, name
        assert torch.equal(edv, dv)
