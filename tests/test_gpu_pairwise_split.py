"""The pairwise kernels on bf16 splits (csrc/pairwise_split.h) at the sizes
where they can go wrong: one past and one short of the tile (64, 128), strip
(256 columns), step (32 rows) and feature (32, 64) edges, odd widths (rows off
any vector boundary, a last column without a pair), M = 1, walks of several
strips whose partial rows are added to, and the tiles that sum the squared
differences directly.

Tolerance, on the 2-norm of the error over the 2-norm of the float64 result:
a split product is exact in the matrix unit's input, so an output is off by
the roundings of its accumulation, at most six for 32 terms, of relative size
2^-24 and independent, and a few of its epilogue: 2^-24 (4 + sqrt(6 ceil(k /
32))), k the longest contraction (D, N or M).
"""

import math

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import cosine_sim as oc
from oracle import rbf as orbf

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (64, 128, 32), (65, 127, 33), (63, 129, 31), (128, 257, 64), (129, 255, 65),
          (31, 256, 63), (33, 258, 100), (97, 1, 64), (40, 3, 20), (200, 513, 66), (300, 511, 129),
          (1025, 1027, 64), (2050, 2304, 64), (1500, 9000, 70), (3000, 9001, 5)]


def _rel(name, got, ref, k):
    got = got.detach().cpu().double().numpy()
    assert got.shape == ref.shape
    tol = 2.0 ** -24 * (4 + math.sqrt(6 * math.ceil(k / 32)))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"  {name}: {err:.2e} of {tol:.2e}")
    assert err <= tol, name


def _inputs(n, m, d, scale):
    g = torch.Generator().manual_seed(n + 3 * m + 7 * d)
    return (torch.randn(n, d, generator=g) * scale, torch.randn(m, d, generator=g) * scale,
            torch.randn(n, m, generator=g))


@pytest.mark.parametrize("n,m,d", SHAPES)
def test_rbf_split_edges(n, m, d):
    announce(f"rbf split n={n} m={m} d={d}")
    from cases.rbf import op
    X, Y, G = _inputs(n, m, d, d ** -0.5)
    Xd, Yd = X.cuda().requires_grad_(True), Y.cuda().requires_grad_(True)
    K = op.candidate({"X": Xd, "Y": Yd}, {"gamma": 0.5})
    dX, dY = torch.autograd.grad(K, [Xd, Yd], G.cuda())
    torch.cuda.synchronize()
    Kr = orbf.forward_f64(X.numpy(), Y.numpy(), 0.5)
    dXr, dYr = orbf.backward_f64(X.numpy(), Y.numpy(), G.numpy(), Kr, 0.5)
    _rel("K", K, Kr, d)
    _rel("dX", dX, dXr, max(n, m, d))
    _rel("dY", dY, dYr, max(n, m, d))


@pytest.mark.parametrize("n,m,d", [s for s in SHAPES if s[2] > 1])
def test_cosine_split_edges(n, m, d):
    announce(f"cosine split n={n} m={m} d={d}")
    from cases.cosine_sim import op
    A, B, G = _inputs(n, m, d, 1.0)
    Ad, Bd = A.cuda().requires_grad_(True), B.cuda().requires_grad_(True)
    S = op.candidate({"A": Ad, "B": Bd}, {"eps": 1e-8})
    dA, dB = torch.autograd.grad(S, [Ad, Bd], G.cuda())
    torch.cuda.synchronize()
    An, Bn, Gn = A.double().numpy(), B.double().numpy(), G.double().numpy()
    dAr, dBr = oc.backward_f64(An, Bn, Gn, 1e-8)
    # the rows are normalised in fp32 first: the roundings of a norm and a scale
    _rel("S", S, oc.forward_f64(An, Bn, 1e-8), max(d, 128))
    _rel("dA", dA, dAr, max(n, m, d, 128))
    _rel("dB", dB, dBr, max(n, m, d, 128))


@pytest.mark.parametrize("n,d", [(150, 100), (130, 20), (300, 40)])
def test_rbf_narrow_kernel_keeps_the_direct_distance(n, d):
    """gamma |x|^2 far past the bound up to which distances come from norms
    and products: the squared differences are summed directly, so K(x, x) is
    exactly 1 and a near pair keeps its distance.  One row of large norm sends
    only its own tiles there."""
    announce(f"rbf direct tiles n={n} d={d}")
    from cases.rbf import op
    X, _, _ = _inputs(n, 1, d, 1.0)
    Y = X + 1e-3 * torch.randn(n, d, generator=torch.Generator().manual_seed(5))
    for gamma, base in ((50.0, X), (0.5 / d, torch.cat([X, 1e3 * X[:1]]))):
        K = op.rbf_forward(base.cuda(), base.cuda(), gamma)
        if gamma == 50.0:
            assert bool((K.diagonal() == 1).all())
            _rel("near", op.rbf_forward(X.cuda(), Y.cuda(), gamma).diagonal(),
                 np.diagonal(orbf.forward_f64(X.numpy(), Y.numpy(), gamma)), d)
        else:
            _rel("K", K, orbf.forward_f64(base.numpy(), base.numpy(), gamma), d)
            assert K[n, n].item() == 1 and bool((K[n, :n] == 0).all())


@pytest.mark.parametrize("d", [64, 40])
def test_rbf_infinite_row(d):
    """A row holding an infinity is at distance infinity: K is 0 there and
    finite everywhere else."""
    announce(f"rbf infinite row d={d}")
    from cases.rbf import op
    X, Y, _ = _inputs(200, 150, d, d ** -0.5)
    Kr = orbf.forward_f64(X.numpy(), Y.numpy(), 0.5)
    X[70, 3] = float("inf")
    Kr[70] = 0.0
    _rel("K", op.rbf_forward(X.cuda(), Y.cuda(), 0.5), Kr, d)
