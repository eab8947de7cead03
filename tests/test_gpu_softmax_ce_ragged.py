"""Softmax cross-entropy on rows of any width and alignment: widths next to the
edges of the row kernels (lanes per row, windows per lane, segments), where the
last window reaches back over the one before, on arrays that start off a
16-byte boundary too.  Against float64: lse within 2^-24 (2 |lse| + 8) (its
max, its logarithm and a sum of C exponentials in a tree), dlogits within a
relative 2^-24 (4 + 2 max |x - lse|) of the exponential's argument."""

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import softmax_ce as osce

pytestmark = pytest.mark.gpu

WIDTHS = [33, 63, 65, 127, 129, 131, 255, 257, 511, 513, 514, 515, 1023, 1025, 2047, 2049, 4095,
          4097, 8191, 8193, 8194, 12289]


def _device(x, off):
    flat = torch.empty(x.numel() + off, device="cuda")
    out = flat[off:].view(x.shape)
    out.copy_(x)
    return out


def _run(x, labels, off):
    from cases.softmax_ce import op
    xd, ld = _device(x, off), labels.cuda()
    loss, lse = op.sce_forward(xd, ld)
    d = op.sce_backward(xd, ld, lse, torch.ones(1, device="cuda"))
    torch.cuda.synchronize()
    return loss, lse, d


@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("c", WIDTHS)
def test_ragged_widths(c, off):
    announce(f"softmax_ce width {c} offset {off}")
    b = 37 if c < 1000 else 9
    g = torch.Generator().manual_seed(c)
    x = torch.randn(b, c, generator=g) * 3
    labels = torch.randint(0, c, (b,), generator=g)
    labels[0], labels[1], labels[2] = 0, c - 1, (c - 1) // 4 * 4 - 1
    loss, lse, d = _run(x, labels, off)
    xd = x.double().numpy()
    ref = np.log(np.exp(xd).sum(1))
    assert np.all(np.abs(lse.cpu().double().numpy() - ref) <= 2.0 ** -24 * (2 * np.abs(ref) + 8))
    want = osce.forward_f64(xd, labels.numpy())
    want = float(np.ravel(want[0] if isinstance(want, tuple) else want)[0])
    assert abs(loss.item() - want) <= 2.0 ** -24 * (4 * abs(want) + 16)
    p = np.exp(xd - ref[:, None])
    p[np.arange(b), labels.numpy()] -= 1
    p /= b
    err = np.abs(d.cpu().double().numpy() - p)
    tol = 2.0 ** -24 * (4 + 2 * np.abs(xd - ref[:, None]).max())
    assert np.all(err <= tol * (np.abs(p) + (1.0 / b) * (p < 0)))


@pytest.mark.parametrize("c", [35, 129, 1001, 8195])
def test_ragged_infinities_and_labels(c):
    """A row of -inf alone has lse = -inf (and a NaN loss), one +inf gives NaN,
    a label outside the row makes its gradient NaN, and no row's values reach
    another through a shared window."""
    announce(f"softmax_ce infinities width {c}")
    x = torch.randn(6, c, generator=torch.Generator().manual_seed(c))
    x[1] = float("-inf")
    x[3, c - 1] = float("inf")
    x[5, : c - 1] = float("-inf")
    labels = torch.tensor([c - 1, 0, c, 1, -1, c - 1])
    loss, lse, d = _run(x, labels, 0)
    lse, d = lse.cpu(), d.cpu()
    assert bool(torch.isnan(loss))
    assert lse[1].item() == float("-inf") and bool(torch.isnan(lse[3]))
    assert bool(torch.isfinite(lse[[0, 2, 4, 5]]).all())
    assert abs(lse[5].item() - x[5, c - 1].item()) < 1e-6
    for r in (1, 2, 3, 4):
        assert bool(torch.isnan(d[r]).all()), r
    for r in (0, 5):
        assert bool(torch.isfinite(d[r]).all()), r
