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
