"""The cuts of the split pairwise kernels (csrc/pairwise_split.h), computed on
the host by a small program built from that header: every shape they accept
keeps the byte offsets of 32 rows of X, W and the partials below 2^31 (the
kernel addresses them with 32 bits), the partials inside the caller's workspace
and the launch below 2^32 threads."""

import os
import shutil
import subprocess

import pytest

from framework import loader

PROGRAM = r"""
#include <cstdio>
#include "pairwise_split.h"
int main() {
  long long n, m, d;
  while (std::scanf("%lld %lld %lld", &n, &m, &d) == 3) {
    const size_t floats = nl2k::pairwise::split_floats(n, m, d, true);
    const auto p = nl2k::pairwise::plan_split_backward(n, m, d, true, floats);
    const auto f = nl2k::pairwise::plan_split_forward(n, m, d);
    std::printf("%d %zu %zu %lld %d %d %lld\n", (int)p.ok, floats, p.ws_floats,
                (long long)p.nRI * p.nRJ, p.n_dc, f.n_jt, (long long)f.n_tiles);
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if not shutil.which(loader.HIPCC) and not os.path.exists(loader.HIPCC):
        pytest.skip("needs hipcc")
    folder = tmp_path_factory.mktemp("plans")
    source, program = folder / "plans.hip", folder / "plans"
    source.write_text(PROGRAM)
    subprocess.run([loader.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I",
                    loader.INCLUDE_DIR, "-I", loader.CSRC_DIR, str(source), "-o", str(program)],
                   check=True)

    def ask(shapes):
        text = "".join("%d %d %d\n" % s for s in shapes)
        out = subprocess.run([str(program)], input=text, check=True, capture_output=True, text=True)
        return [tuple(int(v) for v in line.split()) for line in out.stdout.splitlines()]
    return ask


SIZES = [1, 31, 33, 4096, 100003, 1 << 24, (1 << 24) + 1, 1 << 30]
WIDTHS = [1, 64, 100, 1 << 20, 1 << 24, (1 << 24) + 1, 17_400_000, 25_165_825, 34_600_000,
          67_200_000, (1 << 31) - (1 << 20)]


def test_split_backward_offsets_fit_32_bits(plans):
    shapes = [(n, m, d) for n in SIZES for m in SIZES for d in WIDTHS
              if n * m <= 1 << 36 and n * d <= 1 << 36 and m * d <= 1 << 36]
    for (n, m, d), (ok, floats, used, regions, passes, *_) in zip(shapes, plans(shapes)):
        if not ok:
            continue
        assert 32 * d * 4 <= 1 << 31, (n, m, d)
        assert 32 * m * 4 <= 1 << 31, (n, m, d)
        assert used <= floats, (n, m, d)
        assert -(-regions // 8) * 8 * passes * 512 < 1 << 32, (n, m, d)


def test_split_backward_takes_ordinary_shapes(plans):
    shapes = [(64, 64, 64), (4096, 4096, 64), (1, 1, 1), (3000, 2500, 100), (100000, 7, 3),
              (7, 100000, 300), (8192, 8192, 256), (32, 32, 1 << 24)]
    assert all(p[0] for p in plans(shapes))


def test_split_forward_launches_below_2_32_threads(plans):
    shapes = [(n, m, 1) for n in SIZES + [(1 << 30) + 65] for m in SIZES if n * m <= 1 << 36]
    got = plans(shapes)
    for shape, (*_, n_jt, tiles) in zip(shapes, got):
        assert n_jt == 0 or tiles * 256 < 1 << 32, shape
    assert any(p[-2] == 0 for p in got) and any(p[-2] > 0 for p in got)
