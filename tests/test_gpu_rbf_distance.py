"""The RBF forward's distances where norms and products cancel: identical rows,
near rows, few features, large norms, and D = 64 on and off a 16-byte boundary.

Bound on each entry: K is exp2 of an exponent rounded to fp32 once (2^-24 of
it) and exp2 itself is good to a unit in the last place, so the relative error
is at most 2^-23 + 2^-24 ln(1 / K); the distance is exact beside that.  Where the
squared differences are summed in fp32 (large norms at D = 64) the sum adds D / 2
+ 1 roundings at most, of the exponent.
"""

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _f64(X, Y, gamma):
    d = X.double().numpy()[:, None, :] - Y.double().numpy()[None, :, :]
    return np.exp(-gamma * (d * d).sum(-1))


def _put(X, misaligned):
    """X on the GPU, its first row 4 bytes past a 16-byte boundary if asked."""
    if not misaligned:
        return X.cuda()
    return torch.cat([torch.zeros(1), X.flatten()]).cuda()[1:].view_as(X)


def _entries(name, K, ref, fp32_terms=0):
    got = K.cpu().double().numpy()
    keep = ref > 1e-37
    e = -np.log(ref[keep])
    rel = np.abs(got[keep] - ref[keep]) / ref[keep]
    tol = 2.0 ** -23 + 2.0 ** -24 * e * (1 + fp32_terms)
    print(f"  {name}: worst {np.max(rel / tol):.2f} of the bound, {rel.max():.2e}")
    assert np.all(rel <= tol), name
    assert np.all(got[~keep] <= 1e-36), name


@pytest.mark.parametrize("d,misaligned", [(1, False), (4, False), (7, False), (16, False),
                                          (40, False), (63, False), (64, True), (65, True),
                                          (100, False), (130, True)])
@pytest.mark.parametrize("level", [0.5, 4.0, 400.0])
def test_rbf_distances(d, misaligned, level):
    """gamma |x|^2 about `level`: rows against themselves, against rows 1 %
    apart, and against unrelated ones."""
    announce(f"rbf distances d={d} misaligned={misaligned} level={level}")
    from cases.rbf import op
    gamma, n = 0.5, 150
    g = torch.Generator().manual_seed(d)
    X = torch.randn(n, d, generator=g) * (level / gamma / d) ** 0.5
    Y = X * (1 + 0.01 * torch.randn(n, d, generator=g))
    Xd, Yd = _put(X, misaligned), _put(Y, misaligned)
    K = op.rbf_forward(Xd, Xd, gamma)
    assert bool((K.diagonal() == 1).all()) and torch.equal(K, K.t().contiguous())
    _entries("rows against themselves", K, _f64(X, X, gamma))
    _entries("near rows", op.rbf_forward(Xd, Yd, gamma), _f64(X, Y, gamma))


@pytest.mark.parametrize("d", [20, 64, 65, 100])
@pytest.mark.parametrize("misaligned", [False, True])
def test_rbf_large_norms(d, misaligned):
    """Features offset by 1000: the distance is a part in 1e6 of the norms."""
    announce(f"rbf large norms d={d} misaligned={misaligned}")
    from cases.rbf import op
    g = torch.Generator().manual_seed(d)
    X = 1000 + torch.randn(140, d, generator=g) * d ** -0.5
    Xd = _put(X, misaligned)
    for gamma in (0.5, 1e-3):
        K = op.rbf_forward(Xd, Xd, gamma)
        assert bool((K.diagonal() == 1).all())
        _entries(f"gamma {gamma}", K, _f64(X, X, gamma), fp32_terms=d / 2 + 1)
