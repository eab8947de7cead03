"""LayerNorm and L2-norm-scale on rows of any width and alignment: widths next
to the edges of the row kernels (16 lanes, a wave, 256, 512 and 1024 threads a
row; whole and cut float4), every operand off a 16-byte boundary too, with the
workspace that the library asks for and with the smaller one that it accepts.
Sentinels around each output stay as they were.

Tolerances, against float64, u = 2^-24: a row sum of D floats is at most 32
serial adds and 10 levels of a tree, so 48 u of the sum of magnitudes; a
column sum of at most B rows (B + 24) u of its magnitudes, on xh that carry
the error of the statistics."""

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
WIDTHS = [1, 2, 3, 5, 7, 61, 63, 64, 65, 66, 127, 129, 130, 255, 257, 511, 513, 767, 769, 1001,
          1023, 1025, 2047, 2049, 4095, 4096, 4097, 8191, 8193, 16382, 16383]


class _Padded:
    """A device array `off` floats past a 16-byte boundary between sentinels."""

    def __init__(self, shape, off, data=None):
        n = int(np.prod(shape))
        self.flat = torch.full((n + off + 64,), 777.0, device="cuda")
        self.off, self.n = 32 + off, n
        self.view = self.flat[self.off:self.off + n].view(shape)
        if data is not None:
            self.view.copy_(data)
        self.ptr = self.view.data_ptr()

    def out(self):
        assert torch.all(self.flat[:self.off] == 777.0)
        assert torch.all(self.flat[self.off + self.n:] == 777.0)
        return self.view.cpu().double().numpy()


def _near(name, got, want, tol):
    err = np.abs(got - want)
    assert np.all(err <= tol), (name, float((err - tol).max()), float((err / tol).max()))


def _run(case, b, d, off, short):
    g = torch.Generator().manual_seed(1000 * d + off)
    x = torch.randn(b, d, generator=g) * 2 + (0.5 if case == "layernorm" else 0)
    w, bias, dy = (torch.randn(*s, generator=g) for s in ((d,), (d,), (b, d)))
    eps = 1e-3
    if case == "layernorm":
        from cases.layernorm import op
    else:
        from cases.l2norm_scale import op
    lib = op._lib()
    X, W, Bi, DY = (_Padded(t.shape, off, t) for t in (x, w, bias, dy))
    Y, DX = _Padded((b, d), off), _Padded((b, d), off)
    S0, S1, DW, DB = _Padded((b,), 0), _Padded((b,), 0), _Padded((d,), 0), _Padded((d,), 0)
    centered = case == "layernorm"
    if centered:
        st = lib.layernorm_forward_f32(X.ptr, W.ptr, Bi.ptr, Y.ptr, S0.ptr, S1.ptr, b, d, eps, None)
        need = lib.layernorm_backward_workspace_bytes(b, d)
    else:
        st = lib.l2norm_scale_forward_f32(X.ptr, W.ptr, Y.ptr, S1.ptr, b, d, eps, None)
        need = lib.l2norm_scale_backward_workspace_bytes(b, d)
    assert st == 0
    # one partial row per 64 columns' share of about 2048 workgroups
    groups = min(max(1, -(-2048 // -(-d // 64))), 512, b)
    size = (2 if centered else 1) * -(-b // -(-b // groups)) * d * 4 if short else need
    WS = _Padded(((size + 3) // 4,), 0)
    if centered:
        st = lib.layernorm_backward_f32(DY.ptr, X.ptr, W.ptr, S0.ptr, S1.ptr, DX.ptr, DW.ptr,
                                        DB.ptr, b, d, WS.ptr, size, None)
    else:
        st = lib.l2norm_scale_backward_f32(DY.ptr, X.ptr, W.ptr, S1.ptr, DX.ptr, DW.ptr, b, d,
                                           WS.ptr, size, None)
    assert st == 0
    torch.cuda.synchronize()
    WS.out()

    x, w, bias, dy = (t.double().numpy() for t in (x, w, bias, dy))
    n = d if centered else 1
    mu = x.mean(1, keepdims=True) if centered else np.zeros((b, 1))
    ss = ((x - mu) ** 2).sum(1, keepdims=True) / n + np.float32(eps).astype(np.float64)
    rs = 1 / np.sqrt(ss)
    xh = (x - mu) * rs
    e_mu = 50 * U * np.abs(x).mean(1, keepdims=True) * centered
    e_xh = 60 * U * np.abs(xh) + (e_mu + 2 * U * np.abs(x)) * rs  # statistics, then the difference
    _near("y", Y.out(), xh * w + bias * centered,
          (e_xh + 4 * U * np.abs(xh)) * np.abs(w) + 2 * U * np.abs(bias))
    if centered:
        _near("mean", S0.out()[:, None], mu, e_mu + U * np.abs(mu))
        _near("rstd", S1.out()[:, None], rs, 60 * U * rs + (e_mu * rs) ** 2 * rs)
    else:
        _near("norm", S1.out()[:, None], 1 / rs, 60 * U / rs)
    gw = dy * w
    mg = gw.mean(1, keepdims=True) * centered
    mgx = (gw * xh).sum(1, keepdims=True) / n
    a_mg = np.abs(gw).mean(1, keepdims=True) * centered
    a_mgx = np.abs(gw * xh).sum(1, keepdims=True) / n
    e_mgx = 52 * U * a_mgx + (np.abs(gw) * e_xh).sum(1, keepdims=True) / n
    dx = rs * (gw - mg - xh * mgx)
    _near("dx", DX.out(), dx,
          rs * (70 * U * (np.abs(gw) + a_mg + np.abs(xh) * a_mgx) + np.abs(xh) * e_mgx
                + e_xh * np.abs(mgx)))
    _near("dw", DW.out(), (dy * xh).sum(0),
          (b + 24) * U * np.abs(dy * xh).sum(0) + (np.abs(dy) * e_xh).sum(0))
    if centered:
        _near("dbias", DB.out(), dy.sum(0), (b + 24) * U * np.abs(dy).sum(0))


@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("d", WIDTHS)
@pytest.mark.parametrize("case", ["layernorm", "l2norm_scale"])
def test_any_width_and_alignment(case, d, off):
    announce(f"{case} width {d} offset {off}")
    _run(case, 1037 if d < 300 else 133, d, off, False)


@pytest.mark.parametrize("case,b,d", [("layernorm", 4, 16383), ("layernorm", 300, 16383),
                                      ("l2norm_scale", 4100, 129), ("l2norm_scale", 2, 7)])
def test_smaller_workspace(case, b, d):
    announce(f"{case} [{b}, {d}] smaller workspace")
    _run(case, b, d, 1, True)


def test_underflowed_norm_keeps_its_infinities():
    """x^2 underflows, eps = 0: the norm is 0, x / norm infinite and dX with it."""
    announce("l2norm_scale underflowed norm")
    from cases.l2norm_scale import op
    x = torch.full((3, 131), 1e-30, device="cuda")
    g = torch.ones(131, device="cuda")
    y, norm = op.l2n_forward(x, g, 0.0)
    dx, _ = op.l2n_backward(x, g, torch.ones_like(x), norm)
    torch.cuda.synchronize()
    assert torch.all(norm == 0) and torch.all(torch.isinf(y)) and torch.all(torch.isinf(dx))
