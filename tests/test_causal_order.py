"""The order of a causal problem's workgroups where the (batch, head) slices do not divide by eight (csrc/causal_order.hpp), compiled
for the host: every unit once, every XCD's share of the work nearly the same and walked from the longest to the shortest."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "causal_order.hpp"
int main(int, char** argv) {
    const int slices = atoi(argv[1]), levels = atoi(argv[2]);
    for (int i = 0; i < slices * levels; ++i) {
        int s = -1, l = -1;
        fattn::causal_order(i, slices, levels, s, l, [](int j, int) { return j; });
        printf("%d %d\n", s, l);
    }
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(d / "order.cpp"), "-o", str(d / "order")], check=True)
    return str(d / "order")


@pytest.mark.parametrize("slices,levels", [(1, 1), (1, 7), (1, 64), (3, 5), (7, 9), (9, 1), (12, 8), (21, 24), (30, 13), (36, 17), (43, 12), (107, 3),
                                           (250, 1040), (260999, 1), (4, 65536)])
def test_order(exe, slices, levels):
    out = subprocess.run([exe, str(slices), str(levels)], check=True, capture_output=True, text=True).stdout.split()
    units = list(zip(map(int, out[::2]), map(int, out[1::2])))
    assert sorted(units) == [(s, v) for s in range(slices) for v in range(levels)]
    work = []
    for x in range(8):
        mine = [v for _, v in units[x::8]]
        # along an XCD's sequence: its own slices level by level, the others among them at most one level (of eight XCDs' steps) off
        run = 0
        for v in mine:
            assert v >= run - 1 - 8 // max(1, slices % 8)
            run = max(run, v)
        work.append(sum(levels - v for v in mine))
        own = [s for s, _ in units[x::8] if s < slices // 8 * 8]
        assert all(s % 8 == x for s in own)
    assert max(work) - min(work) <= 2 * levels       # units of the left-over slices, dealt one by one
