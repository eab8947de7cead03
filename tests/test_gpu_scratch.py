"""Backward calls whose fastest route's workspace does not fit the GPU run with
the least they need (the allocation that fails is asked for in earnest: more
memory than any GPU has)."""

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

HUGE = 1 << 50


def _close(got, want):
    for a, b in zip(got, want):
        assert float((a - b).norm() / b.norm()) <= 1e-6


def test_spmm_backward_without_room(monkeypatch):
    announce("spmm backward, no room for the column buckets")
    from cases.spmv import op
    m, k, d = 900, 20000, 8
    ptr = (torch.arange(m + 1) * 11).int().cuda()
    col = torch.randint(0, k, (11 * m,), generator=torch.Generator().manual_seed(1)).int().cuda()
    vals, X, G = torch.randn(11 * m).cuda(), torch.randn(k, d).cuda(), torch.randn(m, d).cuda()
    want = op.spmv_backward(ptr, col, vals, X, G)
    least = op._lib().spmv_backward_workspace_bytes(m, k, d, 11 * m)
    monkeypatch.setattr(op, "_workspace_bytes", lambda *shape: (HUGE, least))
    _close(op.spmv_backward(ptr, col, vals, X, G), want)


@pytest.mark.parametrize("d", [33, 100])
def test_rbf_backward_without_room(monkeypatch, d):
    announce(f"rbf backward, no room for partials, d={d}")
    from cases.rbf import op
    X, Y, G = torch.randn(300, d).cuda(), torch.randn(500, d).cuda(), torch.randn(300, 500).cuda()
    K = torch.rand(300, 500).cuda()
    want = op.rbf_backward(X, Y, G, K, 0.5)
    monkeypatch.setattr(op, "_workspace_bytes", lambda *shape: HUGE)
    _close(op.rbf_backward(X, Y, G, K, 0.5), want)


@pytest.mark.parametrize("d", [33, 100])
def test_cosine_backward_without_room(monkeypatch, d):
    announce(f"cosine backward, no room for partials, d={d}")
    from cases.cosine_sim import op
    A, B, G = torch.randn(300, d).cuda(), torch.randn(500, d).cuda(), torch.randn(300, 500).cuda()
    inv = [1 / t.norm(dim=1) for t in (A, B)]
    want = op.cos_backward(A, B, *inv, G)
    monkeypatch.setattr(op, "_workspace_bytes", lambda *shape: HUGE)
    _close(op.cos_backward(A, B, *inv, G), want)


@pytest.mark.parametrize("n,m,d", [(300, 500, 33), (64, 64, 100), (2000, 1500, 100)])
def test_cosine_backward_takes_any_workspace_from_the_least(n, m, d):
    announce(f"cosine backward, workspaces from the least, {n} x {m} x {d}")
    from cases.cosine_sim import op
    from framework import capi
    A, B, G = torch.randn(n, d).cuda(), torch.randn(m, d).cuda(), torch.randn(n, m).cuda()
    inv = [1 / t.norm(dim=1) for t in (A, B)]
    want = op.cos_backward(A, B, *inv, G)
    lib, least, best = op._lib(), 4 * (n + m) * d, op._workspace_bytes(n, m, d)
    for size in sorted({least, (least + best) // 2 // 4 * 4, best}):
        guard = torch.full((size // 4 + 64,), 7.0, device="cuda")
        dA, dB = torch.empty_like(A), torch.empty_like(B)
        P = capi.ptr
        st = lib.cosine_sim_backward_f32(P(A), P(B), P(inv[0]), P(inv[1]), P(G), P(dA), P(dB), n, m,
                                         d, P(guard), size, capi.stream_of(A))
        capi.check(st, lib.cosine_sim_last_error, "cos_backward")
        _close((dA, dB), want)
        assert bool((guard[size // 4:] == 7.0).all())
    assert lib.cosine_sim_backward_f32(P(A), P(B), P(inv[0]), P(inv[1]), P(G), P(dA), P(dB), n, m, d,
                                       P(guard), least - 4, capi.stream_of(A)) != 0
