"""The rule that spreads the gather passes over workgroups (dfr_spread.h, plain
C++) over every particle count and domain a context takes: a spread launch stays
within the grid where spreading was measured to pay, so a large, nearly empty
domain runs one workgroup per brick and no launch passes HIP's 2^32 threads where
one workgroup per brick does not.
"""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "difffr_amd", "csrc")
BLOCK = 640        # threads of a workgroup
CELL_PARTS = 8     # most workgroups a brick of the cell-wise list build

MAIN = r"""
#include <cstdio>
#include "dfr_spread.h"
int main() {
  int nf; unsigned nb;
  while (std::scanf("%d %u", &nf, &nb) == 2) std::printf("%d\n", dfr::gather_parts_log2(nf, nb));
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("spread")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "rule")],
                   check=True)

    def ask(pairs):
        text = "".join(f"{n} {b}\n" for n, b in pairs)
        out = subprocess.run([str(d / "rule")], input=text, capture_output=True, text=True, check=True).stdout
        return [int(v) for v in out.split()]

    return ask


COUNTS = [0, 1, 500, 2000, 16383, 16384, 39999, 40000, 44000, 60000, 79999, 80000, 1000000, 4000000]
BRICKS = [1, 64, 500, 1280, 1281, 2560, 2561, 9261, 117649, 838860, 838861, 6710886]


def test_spread_grids_are_bounded(rule):
    pairs = [(n, b) for n in COUNTS for b in BRICKS]
    for (n, b), parts in zip(pairs, rule(pairs)):
        assert 0 <= parts <= 2
        assert parts == 0 or (b << parts) <= 5120, (n, b)
        assert parts == 0 or b * CELL_PARTS * BLOCK < 2 ** 32, (n, b)
        assert n < 80000 or parts == 0, (n, b)


def test_full_small_tanks_are_spread(rule):
    assert rule([(1000, 64), (8000, 175), (28000, 336), (60000, 500), (100000, 900)]) == [2, 2, 2, 1, 0]


def test_sparse_domains_are_not(rule):
    assert rule([(1000, 4913), (2000, 9261), (30000, 117649), (1000, 6710886)]) == [0, 0, 0, 0]
