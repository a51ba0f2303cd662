"""How a launch's workgroups take a work list (frk_deal.hpp): every entry once, every XCD (block id mod 8) the same
number of them to within one, neighbouring entries together."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include <cstdio>
#include <cstdlib>
#include "frink_amd/csrc/frk_deal.hpp"
int main(int, char **argv) {
    const int n = atoi(argv[1]);
    for (int b = 0; b < frk::deal_grid(n); b++) printf("%d ", frk::deal_entry(b, n));
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("deal")
    (d / "deal.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-I", ROOT, str(d / "deal.cpp"), "-o", str(d / "deal")])
    return lambda n: [int(v) for v in subprocess.check_output([str(d / "deal"), str(n)]).split()]


# 18 row tiles x 2 token tiles x 6 parts: dealt by row tile, two XCDs had 36 workgroups for their 32 CUs
@pytest.mark.parametrize("entries", [1, 7, 8, 9, 40, 216, 255, 256, 257, 1000, 4099])
def test_every_xcd_has_an_equal_run(deal, entries):
    taken = deal(entries)
    assert sorted(e for e in taken if e >= 0) == list(range(entries))
    runs = [[e for e in taken[x::8] if e >= 0] for x in range(8)]
    for run in runs:
        assert run == list(range(run[0], run[0] + len(run))) if run else True
        assert len(run) in (entries // 8, -(-entries // 8))
