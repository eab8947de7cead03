"""Softmax cross-entropy past the limits of its launches, and rows of
infinities."""

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def test_backward_more_segments_than_a_launch():
    """More ragged rows than a launch has workgroups of 256 threads: slices of
    the gradient against float64.  An entry is the product of four numbers and
    an exponential whose argument, up to 16, is rounded twice."""
    b, c = (1 << 24) + 3, 513
    announce(f"softmax_ce backward [{b}, {c}]")
    from cases.softmax_ce import op
    if torch.cuda.mem_get_info()[0] < 90 << 30:
        pytest.skip("needs 90 GB")
    g = torch.Generator("cuda").manual_seed(1)
    x = torch.randn(b, c, device="cuda", generator=g)
    lab = torch.randint(0, c, (b,), device="cuda", generator=g)
    _, lse = op.sce_forward(x, lab)
    dx = op.sce_backward(x, lab, lse, torch.tensor(float(b), device="cuda"))
    for s in (slice(0, 512), slice(b // 2, b // 2 + 512), slice(b - 512, b)):
        ref = torch.softmax(x[s].double(), 1)
        ref.scatter_add_(1, lab[s, None], torch.full((512, 1), -1.0, dtype=ref.dtype,
                                                     device="cuda"))
        assert float((dx[s].double() - ref).abs().max()) <= 2.0 ** -24 * 2 * (16 + 4)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("c", [1, 7, 12, 13, 31, 32, 33, 100, 1024, 1025, 8193, 50257])
def test_rows_of_infinities(c, offset):
    """At every width, as torch.logsumexp: a row of -inf has lse = -inf, one NaN
    among -inf gives NaN, one finite logit among -inf gives that logit."""
    announce(f"softmax_ce rows of -inf, width {c}, offset {offset}")
    from cases.softmax_ce import op
    b = 70
    x = torch.full((b, c), float("-inf"))
    x[2, c // 2] = float("nan")
    x[3] = float("nan")
    x[4, c - 1] = 2.5
    x[5:] = torch.randn(b - 5, c, generator=torch.Generator().manual_seed(c))
    flat = torch.zeros(b * c + offset, device="cuda")
    xd = flat[offset:].view(b, c)
    xd.copy_(x)
    loss, lse = op.sce_forward(xd, torch.zeros(b, dtype=torch.int64, device="cuda"))
    want = torch.logsumexp(x.double(), 1)
    assert bool(torch.isnan(loss))
    assert torch.allclose(lse.cpu().double(), want, rtol=1e-6, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("b,c", [(3000, 513), (700, 1029), (300, 2051), (64, 50257), (500, 4096),
                                 (500, 100)])
def test_backward_in_place(b, c):
    """The gradient written over the logits, by whichever kernel."""
    announce(f"softmax_ce backward in place [{b}, {c}]")
    from cases.softmax_ce import op
    from framework import capi
    g = torch.Generator("cuda").manual_seed(c)
    x = torch.randn(b, c, device="cuda", generator=g)
    lab = torch.randint(0, c, (b,), device="cuda", generator=g)
    _, lse = op.sce_forward(x, lab)
    one = torch.ones(1, device="cuda")
    want = op.sce_backward(x, lab, lse, one)
    lib, P = op._lib(), capi.ptr
    st = lib.softmax_ce_backward_f32(P(x), P(lab), P(lse), P(one), P(x), b, c, capi.stream_of(x))
    capi.check(st, lib.softmax_ce_last_error, "sce_backward")
    assert torch.allclose(x, want, rtol=1e-6, atol=1e-12)
