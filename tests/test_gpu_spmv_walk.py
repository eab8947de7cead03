"""The D = 1 forward's walk where it can go wrong: rows that start at the edges
of its steps of 256 positions and of its window of 512 row starts, more row
starts in a step than lanes, runs of empty rows around the window's length,
rows longer than many steps.  Values and x are small integers, so every sum is
exact in fp32 whatever its order, and y is compared bit for bit; with the copy
of the gathered x too.  The backward's column sums likewise, over tile counts
that split differently between waves."""

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _rows():
    g = np.random.default_rng(5)
    gaps = []
    for n in (1, 3, 62, 63, 64, 65, 255, 256, 257, 510, 511, 512, 513, 1023, 1024, 1025):
        gaps += [int(g.integers(1, 9))] + [0] * n
    return {
        "one row": [1000],
        "one entry": [0] * 700 + [1] + [0] * 700,
        "ones": [1] * 5000,
        "ones and zeros": [1, 0] * 4000,
        "many starts at a position": ([0] * 70 + [1]) * 300,
        "gaps": gaps,
        "step edges": [255, 256, 257, 1, 255, 0, 0, 512, 3, 4, 5, 252, 1024] * 20,
        "long": [5, 0, 300_000, 0, 0, 7] + [2] * 3000 + [70_001, 1],
        "power law": np.minimum(g.zipf(1.6, 30_000) - 1, 20_000).tolist(),
    }


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("cut", [0, 1, 3])
@pytest.mark.parametrize("name", sorted(_rows()))
def test_forward_walk(name, cut, idx):
    from cases.spmv import op
    announce(f"spmv walk {name} cut {cut} {idx}")
    lens = np.asarray(_rows()[name], np.int64)
    lens[-1] += cut  # nnz modulo 4: the last waves take the scalar loads
    ptr = np.concatenate([[0], np.cumsum(lens)])
    g = np.random.default_rng(lens.size)
    k = 3001
    col = g.integers(0, k, ptr[-1])
    vals = g.integers(-4, 5, ptr[-1]).astype(np.float32)
    x = g.integers(-4, 5, (k, 1)).astype(np.float32)
    rows = np.repeat(np.arange(lens.size), lens)
    want = np.zeros(lens.size)
    np.add.at(want, rows, vals.astype(np.float64) * x[col, 0])  # below 2^24 throughout
    args = (torch.from_numpy(ptr).to(idx).cuda(), torch.from_numpy(col).to(idx).cuda(),
            torch.from_numpy(vals).cuda(), torch.from_numpy(x).cuda())
    y = op.spmv_forward(*args)
    y2, kept = op.spmv_forward(*args, keep_gather=True)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy()[:, 0], want)
    assert np.array_equal(y2.cpu().numpy()[:, 0], want)
    assert np.array_equal(kept.cpu().numpy().ravel(), x[col, 0])


@pytest.mark.parametrize("k", [1, 300, 70_000])
@pytest.mark.parametrize("tiles", [1, 3, 15, 16, 17, 33, 65, 1030])
def test_column_sums_over_tiles(tiles, k):
    """dX where the waves of a bucket's workgroup share a tile of 8192 entries
    (up to 15), take one to 64 tiles each, and take more than one group."""
    from cases.spmv import op
    announce(f"spmv column sums of {tiles} tiles, K={k}")
    nnz, m = 8192 * tiles - 5, 999
    g = np.random.default_rng(tiles)
    ptr = np.sort(np.concatenate([[0, nnz], g.integers(0, nnz + 1, m - 1)]))
    col = g.integers(0, k, nnz)
    vals = g.integers(-1, 2, nnz).astype(np.float32)
    dy = g.integers(-1, 2, (m, 1)).astype(np.float32)
    x = g.integers(-4, 5, (k, 1)).astype(np.float32)
    rows = np.repeat(np.arange(m), np.diff(ptr))
    want = np.bincount(col, weights=vals.astype(np.float64) * dy[rows, 0], minlength=k)
    dv, dx = op.spmv_backward(*(torch.from_numpy(t).cuda() for t in (ptr, col, vals, x, dy)))
    torch.cuda.synchronize()
    assert np.array_equal(dx.cpu().numpy()[:, 0], want)
    assert np.array_equal(dv.cpu().numpy().ravel(), dy[rows, 0] * x[col, 0])
