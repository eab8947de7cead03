"""The pairwise cases past the limits of their tile kernels (32-bit offsets,
workgroups of a launch), on the general kernels.  Against float64; the bound on the 2-norm error is 2^-24 (4 +
sqrt(k)), k the contraction of a sequential sum."""

import math

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _close(name, got, ref_of, width, k, step=1 << 20):
    """got [rows, width] against ref_of(slice of features), in float64."""
    num = den = 0.0
    for c in range(0, width, step):
        s = slice(c, min(c + step, width))
        ref = ref_of(s)
        num += float((got[:, s].double() - ref).square().sum())
        den += float(ref.square().sum())
    err, tol = math.sqrt(num / den), 2.0 ** -24 * (4 + math.sqrt(k))
    print(f"  {name}: {err:.2e} of {tol:.2e}")
    assert err <= tol, name


def _rows(n, d, seed):
    return torch.randn(n, d, device="cuda", generator=torch.Generator("cuda").manual_seed(seed))


# 32 rows of this many features pass 3 GiB, the largest buffer resource used
WIDE = 25_200_004


def test_rbf_backward_wide_features():
    announce(f"rbf backward n=32 m=32 d={WIDE}")
    from cases.rbf import op
    n, d, gamma = 32, WIDE, 0.25
    X, Y, G, K = _rows(n, d, 1), _rows(n, d, 2), _rows(n, n, 3), _rows(n, n, 4).sigmoid()
    dX, dY = op.rbf_backward(X, Y, G, K, gamma)
    W = G.double() * K.double()
    for name, got, A, B, w in (("dX", dX, X, Y, W), ("dY", dY, Y, X, W.t().contiguous())):
        _close(name, got, lambda s: -2 * gamma * (w.sum(1, keepdim=True) * A[:, s].double()
                                                  - w @ B[:, s].double()), d, n)


def test_cosine_backward_wide_features():
    announce(f"cosine backward n=32 m=32 d={WIDE}")
    from cases.cosine_sim import op
    n, d = 32, WIDE
    A, B, G = _rows(n, d, 1), _rows(n, d, 2), _rows(n, n, 3)
    na, nb = (torch.stack([r.double().norm() for r in t]) for t in (A, B))
    ia, ib = (1 / na).float(), (1 / nb).float()
    dA, dB = op.cos_backward(A, B, ia, ib, G)
    for name, got, P, Q, ip, iq, w in (("dA", dA, A, B, ia, ib, G.double()),
                                       ("dB", dB, B, A, ib, ia, G.double().t().contiguous())):
        dot = torch.zeros(n, 1, dtype=torch.float64, device="cuda")
        ip, iq = ip.double()[:, None], iq.double()[:, None]

        def part(s):
            return P[:, s].double() * ip, w @ (Q[:, s].double() * iq)

        for c in range(0, d, 1 << 20):
            ph, acc = part(slice(c, c + (1 << 20)))
            dot += (ph * acc).sum(1, keepdim=True)

        def ref(s):
            ph, acc = part(s)
            return ip * (acc - dot * ph)
        _close(name, got, ref, d, n + d / 64 / 4)


# more outputs in a row than a launch has tiles of 64 columns
TALL = ((1 << 24) << 6) + 5


def _slices(width):
    return [slice(0, 4096), slice(width // 2, width // 2 + 4096), slice(width - 4096, width)]


@pytest.mark.parametrize("turned", [False, True])
def test_rbf_forward_more_tiles_than_a_launch(turned):
    announce(f"rbf forward {TALL} outputs, turned={turned}")
    from cases.rbf import op
    x, Y = _rows(1, 1, 1), _rows(TALL, 1, 2)
    K = op.rbf_forward(Y, x, 0.5) if turned else op.rbf_forward(x, Y, 0.5)
    K = K.flatten()
    for s in _slices(TALL):
        ref = torch.exp(-0.5 * (x[0].double() - Y[s, 0].double()).square())
        assert float((K[s].double() - ref).norm() / ref.norm()) <= 2.0 ** -21


def test_cosine_forward_more_tiles_than_a_launch():
    announce(f"cosine forward {TALL} outputs")
    from cases.cosine_sim import op
    a, B = _rows(1, 2, 1), _rows(TALL, 2, 2)
    S, inv_a, inv_b = op.cos_forward(a, B, 1e-8)
    for s in _slices(TALL):
        b, inv = B[s].double(), 1 / (B[s].double().norm(dim=1) + 1e-8)
        ref = (b * inv[:, None]) @ (a[0].double() / (a.double().norm() + 1e-8))
        assert float((S[0, s].double() - ref).norm() / ref.norm()) <= 2.0 ** -21
        assert float((inv_b[s].double() - inv).norm() / inv.norm()) <= 2.0 ** -21


# more columns than the split backwards take: the general kernels, one side's
# walk in slices and the other's whole
@pytest.mark.parametrize("n", [1, 70])
def test_rbf_backward_many_columns(n):
    m, d, gamma = (1 << 24) + 101, 2, 0.25
    announce(f"rbf backward n={n} m={m} d={d}")
    from cases.rbf import op
    X, Y, G, K = _rows(n, d, 1), _rows(m, d, 2), _rows(n, m, 3), _rows(n, m, 4).sigmoid_()
    dX, dY = op.rbf_backward(X, Y, G, K, gamma)
    acc = torch.zeros(n, d + 1, dtype=torch.float64, device="cuda")
    for c in range(0, m, 1 << 20):
        s = slice(c, min(c + (1 << 20), m))
        W, y = G[:, s].double() * K[:, s].double(), Y[s].double()
        acc[:, d] += W.sum(1)
        acc[:, :d] += W @ y
        wt = W.t().contiguous()
        ref = -2 * gamma * (W.sum(0)[:, None] * y - wt @ X.double())
        assert float((dY[s].double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * (4 + math.sqrt(n))
    ref = -2 * gamma * (acc[:, d:] * X.double() - acc[:, :d])
    # a slice is a sequential sum of 16400 columns, of which there are 1024
    assert float((dX.double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * (4 + math.sqrt(m / 1024))


@pytest.mark.parametrize("n", [1, 70])
def test_cosine_backward_many_columns(n):
    m, d = (1 << 24) + 101, 2
    announce(f"cosine backward n={n} m={m} d={d}")
    from cases.cosine_sim import op
    A, B, G = _rows(n, d, 1), _rows(m, d, 2), _rows(n, m, 3)
    ia, ib = (1 / t.double().norm(dim=1) for t in (A, B))
    dA, dB = op.cos_backward(A, B, ia.float(), ib.float(), G)
    ah, acc = A.double() * ia[:, None], torch.zeros(n, d, dtype=torch.float64, device="cuda")
    for c in range(0, m, 1 << 20):
        s = slice(c, min(c + (1 << 20), m))
        w, bh = G[:, s].double(), B[s].double() * ib[s, None]
        acc += w @ bh
        part = w.t().contiguous() @ ah
        ref = ib[s, None] * (part - (bh * part).sum(1, keepdim=True) * bh)
        # the projection leaves one of two dimensions: its error is the contraction's
        scale = (ib[s, None] * part).norm()
        assert float((dB[s].double() - ref).norm() / scale) <= 2.0 ** -24 * (8 + math.sqrt(n))
    ref = ia[:, None] * (acc - (ah * acc).sum(1, keepdim=True) * ah)
    assert float((dA.double() - ref).norm() / (ia[:, None] * acc).norm()) <= \
        2.0 ** -24 * (8 + math.sqrt(m / 1024))
