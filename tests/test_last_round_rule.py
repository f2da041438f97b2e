"""When 256-query workgroups are not taken for their thin last round (csrc/last_round.hpp): compiled for the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "last_round.hpp"
int main(int argc, char** argv) {
    for (int i = 1; i + 2 < argc; i += 3) printf("%d ", (int)fattn::thin_last_round(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2])));
}
"""


def test_rule(tmp_path):
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    # whole rounds are not thin; up to half (a third) of the units used in the last round is
    cases = [((256, 256, 2), 0), ((512, 256, 3), 0), ((257, 256, 2), 1), ((384, 256, 2), 1), ((385, 256, 2), 0), ((341, 256, 3), 1),
             ((342, 256, 3), 0), ((1, 256, 2), 1), ((200, 256, 2), 0)]
    out = subprocess.run([str(exe), *(str(x) for c, _ in cases for x in c)], check=True, capture_output=True, text=True).stdout.split()
    assert [int(x) for x in out] == [w for _, w in cases]
