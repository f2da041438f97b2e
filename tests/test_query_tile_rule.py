"""Which calls 256-query and which 128-query workgroups serve (csrc/query_tile.hpp), on both sides of every line: compiled for the
host, for 256 compute units."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "query_tile.hpp"
int main(int argc, char** argv) {
    for (int i = 1; i + 6 < argc; i += 7) {
        const char* what = argv[i];
        const long long slices = atoll(argv[i + 1]), q = atoll(argv[i + 2]), k = atoll(argv[i + 3]), d = atoll(argv[i + 4]), causal = atoll(argv[i + 5]), lens = atoll(argv[i + 6]);
        const long long total = (q + 255) / 256 * slices;
        printf("%d ", (int)(!strcmp(what, "fwd")  ? fattn::fwd_takes_256(total, 256, slices, q, k, d == 64 ? 64 : 128, d == 96, causal, lens)
                            : !strcmp(what, "dq") ? fattn::dq_takes_256(total, 256, q, k, d, causal, lens)
                                                  : fattn::sage_takes_256(total, 256, k)));
    }
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(d / "rule.cpp"), "-o", str(d / "rule")], check=True)
    return str(d / "rule")


# slices, queries, keys, head dim, causal, key lengths -> 256
FWD = [  # nothing excluded: one round; an eighth, a half, more of the last round; whole rounds; a handful more than whole rounds
    ((64, 1024, 1024, 64, 0, 0), 1), ((72, 1024, 768, 64, 0, 0), 0), ((72, 1024, 832, 128, 0, 0), 1), ((68, 1024, 1024, 128, 0, 0), 1), ((136, 1024, 1024, 128, 0, 0), 0),
    ((136, 1024, 1088, 128, 0, 0), 1), ((80, 1024, 2048, 128, 0, 0), 0), ((160, 1024, 2112, 128, 0, 0), 1), ((84, 1024, 2112, 128, 0, 0), 0), ((96, 1024, 2112, 128, 0, 0), 1),
    ((96, 1024, 3072, 64, 0, 0), 0), ((96, 1024, 3136, 64, 0, 0), 1), ((112, 1024, 512, 128, 0, 0), 0), ((112, 1024, 576, 128, 0, 0), 1), ((112, 1024, 1024, 64, 0, 0), 0),
    ((112, 1024, 1088, 64, 0, 0), 1), ((66, 1024, 512, 64, 0, 0), 1), ((96, 1024, 512, 96, 0, 0), 1), ((80, 1024, 512, 96, 0, 0), 0),
    # the last key tile cut
    ((64, 1024, 1011, 128, 0, 0), 1), ((64, 1024, 1011, 64, 0, 0), 0), ((66, 1024, 499, 128, 0, 0), 0), ((112, 1024, 499, 128, 0, 0), 0), ((112, 1024, 1011, 128, 0, 0), 1),
    ((96, 1024, 2035, 128, 0, 0), 0), ((96, 1024, 2100, 128, 0, 0), 1), ((72, 1024, 2100, 128, 0, 0), 0),
    # causal: short, one round, more, slices that do not divide by eight; the second round full
    ((96, 768, 768, 128, 1, 0), 0), ((128, 768, 768, 128, 1, 0), 1), ((64, 1024, 1024, 128, 1, 0), 0), ((64, 1024, 1088, 128, 1, 0), 1), ((16, 4096, 4096, 128, 1, 0), 0),
    ((24, 4096, 4096, 128, 1, 0), 1), ((32, 4096, 4096, 128, 1, 0), 1), ((28, 4096, 4096, 128, 1, 0), 0), ((128, 1024, 1024, 128, 1, 0), 0), ((80, 1536, 1536, 128, 1, 0), 1),
    ((72, 1536, 1536, 128, 1, 0), 0), ((85, 1536, 1536, 128, 1, 0), 0), ((64, 2048, 2048, 128, 1, 0), 1), ((56, 2048, 2048, 128, 1, 0), 0), ((40, 3072, 3072, 128, 1, 0), 1),
    ((32, 3072, 3072, 128, 1, 0), 0), ((128, 3072, 3072, 128, 1, 0), 0), ((21, 6144, 6144, 128, 1, 0), 1), ((14, 8192, 8192, 128, 1, 0), 1), ((12, 8192, 8192, 128, 1, 0), 0),
    ((20, 8192, 8192, 128, 1, 0), 0), ((7, 16384, 16384, 128, 1, 0), 1), ((9, 12288, 12288, 128, 1, 0), 0), ((64, 2048, 2048, 64, 1, 0), 0), ((40, 3072, 3072, 96, 1, 0), 1),
    # key lengths: where the last round allows it
    ((128, 1024, 512, 128, 0, 1), 1), ((132, 1024, 512, 128, 0, 1), 0)]
DQ = [((64, 1024, 512, 128, 0, 0), 1), ((128, 1024, 1024, 128, 0, 0), 0), ((128, 1024, 1088, 128, 0, 0), 1), ((96, 1024, 1088, 128, 0, 0), 0), ((112, 1024, 1088, 128, 0, 0), 1),
      ((192, 1024, 1536, 128, 0, 0), 0), ((192, 1024, 1600, 128, 0, 0), 1), ((136, 1024, 1088, 128, 0, 0), 1), ((192, 1024, 2048, 64, 0, 0), 0), ((192, 1024, 2112, 64, 0, 0), 1),
      ((160, 1024, 3072, 64, 0, 0), 0), ((160, 1024, 3136, 64, 0, 0), 1), ((59, 3072, 3072, 64, 0, 0), 1), ((192, 1024, 1536, 96, 0, 0), 1), ((192, 1024, 1024, 96, 0, 0), 0),
      ((64, 1024, 1024, 128, 1, 0), 0), ((64, 1024, 1088, 128, 1, 0), 1), ((128, 768, 768, 128, 1, 0), 0), ((256, 512, 512, 128, 1, 0), 1), ((64, 3072, 3072, 128, 1, 0), 0),
      ((32, 4096, 4096, 128, 1, 0), 1), ((16, 4096, 4096, 128, 1, 0), 0), ((32, 4096, 4096, 64, 1, 0), 0), ((16, 8192, 8192, 64, 1, 0), 1), ((20, 8192, 8192, 64, 1, 0), 0),
      ((64, 1024, 1024, 96, 1, 0), 1), ((128, 1024, 1088, 128, 0, 1), 1), ((132, 1024, 1088, 128, 0, 1), 0)]
SAGE = [((64, 1024, 512, 128, 0, 0), 1), ((72, 1024, 1024, 128, 0, 0), 0), ((72, 1024, 1088, 128, 0, 0), 1), ((112, 1024, 512, 128, 0, 0), 1), ((160, 1024, 1024, 64, 0, 0), 0)]


@pytest.mark.parametrize("what,cases", [("fwd", FWD), ("dq", DQ), ("sage", SAGE)])
def test_lines(exe, what, cases):
    out = subprocess.run([exe, *(str(x) for c, _ in cases for x in (what, *c))], check=True, capture_output=True, text=True).stdout.split()
    assert [(c, int(x)) for (c, _), x in zip(cases, out)] == [(c, w) for c, w in cases]
