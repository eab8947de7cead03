"""The pairwise backwards at the ends of the fp32 range: infinities, NaN and
numbers near the largest in one entry of the upstream gradient or one row
(the same infinities and NaN as fp32 arithmetic gives, everything else as
before), and operands so small that a third bf16 term of theirs would lie below
bf16's least normal number.

Bound, on the 2-norm error over the finite entries: as for ordinary inputs,
2^-24 (4 + sqrt(6 ceil(k / 32))), k the longest contraction.
"""

import math

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

SHAPES = [(300, 511, 129), (700, 513, 64), (2050, 2304, 64), (200, 1, 33)]


def _inputs(n, m, d):
    g = torch.Generator().manual_seed(n + m + d)
    return (torch.randn(n, d, generator=g), torch.randn(m, d, generator=g),
            torch.randn(n, m, generator=g))


def _dot(W, B):
    """W @ B in float64, products and sums of infinities as they come."""
    return torch.stack([(W * B[:, c]).sum(1) for c in range(B.shape[1])], 1)


def _same(name, got, ref, k):
    got = got.cpu()
    want = ref.float()
    assert torch.equal(torch.isnan(got), torch.isnan(want)), f"{name}: NaN elsewhere"
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf]), name
    # numbers near the largest stand apart: they would hide the others
    finite = torch.isfinite(want)
    for part in (finite & (want.abs() < 1e15), finite & (want.abs() >= 1e15)):
        if part.any():
            scale = want[part].abs().max().double()
            err = (got[part].double() - ref[part]).div(scale).norm()
            err = float(err / ref[part].div(scale).norm())
            tol = 2.0 ** -24 * (4 + math.sqrt(6 * math.ceil(k / 32)))
            print(f"  {name}: {err:.2e} of {tol:.2e}")
            assert err <= tol, name


def _rbf(X, Y, G, K, gamma, k):
    from cases.rbf import op
    dX, dY = op.rbf_backward(X.cuda(), Y.cuda(), G.cuda(), K.cuda(), gamma)
    W = (G * K).double()  # rounded to fp32 once
    for name, got, A, B, w in (("dX", dX, X, Y, W), ("dY", dY, Y, X, W.t().contiguous())):
        A, B = A.double(), B.double()
        _same(name, got, -2 * gamma * (w.sum(1, keepdim=True) * A - _dot(w, B)), k)


VALUES = {"inf": math.inf, "-inf": -math.inf, "nan": math.nan, "past bf16": 3.399e38,
          "2^120": 2.0 ** 120}


@pytest.mark.parametrize("n,m,d", SHAPES)
@pytest.mark.parametrize("value", VALUES)
def test_rbf_backward_extreme_entries(n, m, d, value):
    announce(f"rbf backward n={n} m={m} d={d}, one entry {value}")
    X, Y, G = _inputs(n, m, d)
    X, Y = X / 16, Y / 16  # past bf16 times these stays finite
    K = torch.rand(n, m, generator=torch.Generator().manual_seed(1))
    i, j = n // 3, m // 2
    G[i, j], K[i, j] = VALUES[value], 1.0
    X[i], Y[j] = X[i] / 1024, Y[j] / 1024
    _rbf(X, Y, G, K, 0.25, max(n, m, d))


@pytest.mark.parametrize("n,m,d", SHAPES)
def test_rbf_backward_infinite_feature(n, m, d):
    announce(f"rbf backward n={n} m={m} d={d}, an infinite feature")
    X, Y, G = _inputs(n, m, d)
    K = torch.rand(n, m, generator=torch.Generator().manual_seed(1))
    K[n // 2] = 0  # as the forward gives at an infinite distance
    X[n // 2, d - 1] = math.inf
    _rbf(X, Y, G, K, 0.25, max(n, m, d))


@pytest.mark.parametrize("n,m,d", SHAPES)
@pytest.mark.parametrize("g,k,x", [(-120, 0, 0), (-60, -55, 0), (0, 0, -114)])
def test_rbf_backward_small_operands(n, m, d, g, k, x):
    """dK about 2^g, K about 2^k, features about 2^x; the outputs are kept normal
    by gamma."""
    announce(f"rbf backward n={n} m={m} d={d}, 2^{g} 2^{k} 2^{x}")
    from cases.rbf import op
    X, Y, G = _inputs(n, m, d)
    K = 0.5 + torch.rand(n, m, generator=torch.Generator().manual_seed(1)) / 2
    gamma = 2.0 ** min(120, -(g + k + x))
    args = [(t.double() * 2.0 ** e).float() for t, e in ((X, x), (Y, x), (G, g), (K, k))]
    got = op.rbf_backward(*(t.cuda() for t in args), gamma)
    X, Y, G, K = (t.double() for t in args)
    W = G * K
    for name, o, A, B, w in (("dX", got[0], X, Y, W), ("dY", got[1], Y, X, W.t().contiguous())):
        _same(name, o, -2 * gamma * (w.sum(1, keepdim=True) * A - _dot(w, B)), max(n, m, d))


def _cosine_check(A, B, G, k):
    from cases.cosine_sim import op
    norms = [t.double().norm(dim=1) for t in (A, B)]
    inv = [(1 / v).float() for v in norms]
    dA, dB = op.cos_backward(A.cuda(), B.cuda(), inv[0].cuda(), inv[1].cuda(), G.cuda())
    w = G.double()
    for name, got, P, Q, ip, iq, wt in (("dA", dA, A, B, inv[0], inv[1], w),
                                        ("dB", dB, B, A, inv[1], inv[0], w.t().contiguous())):
        ph = P.double() * ip.double()[:, None]
        acc = _dot(wt, Q.double() * iq.double()[:, None])
        dot = (ph * acc).sum(1, keepdim=True)
        _same(name, got, ip.double()[:, None] * (acc - dot * ph), k)


@pytest.mark.parametrize("n,m,d", [s for s in SHAPES if s[2] != 33])
@pytest.mark.parametrize("value", ["inf", "-inf", "nan", "2^120"])
def test_cosine_backward_extreme_entries(n, m, d, value):
    announce(f"cosine backward n={n} m={m} d={d}, one entry {value}")
    A, B, G = _inputs(n, m, d)
    G[n // 3, m // 2] = VALUES[value]
    if value == "2^120":
        _cosine_check(A, B, G, max(n, m, d))
        return
    from cases.cosine_sim import op
    inv = [(1 / t.double().norm(dim=1)).float().cuda() for t in (A, B)]
    got = op.cos_backward(A.cuda(), B.cuda(), *inv, G.cuda())
    G[n // 3, m // 2] = 0
    want = op.cos_backward(A.cuda(), B.cuda(), *inv, G.cuda())
    for row, o, ref in ((n // 3, got[0], want[0]), (m // 2, got[1], want[1])):
        # dot and row both hold infinities: their difference is not a number
        assert not torch.isfinite(o[row]).any()
        o[row] = ref[row]
        assert torch.equal(o, ref)


@pytest.mark.parametrize("n,m,d", [s for s in SHAPES if s[2] != 33])
@pytest.mark.parametrize("g", [-118, -100])
def test_cosine_backward_small_gradient(n, m, d, g):
    announce(f"cosine backward n={n} m={m} d={d}, 2^{g}")
    A, B, G = _inputs(n, m, d)
    # rows of length about 1/64, so that the outputs stay normal numbers
    _cosine_check(A / 512, B / 512, (G.double() * 2.0 ** g).float(), max(n, m, d))
