"""Which keep-masks are turned into bits (csrc/mask_route.hpp): compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "mask_route.hpp"
int main(int argc, char** argv) {
    for (int i = 1; i + 7 < argc; i += 8) {
        long long a[8];
        for (int j = 0; j < 8; ++j) a[j] = atoll(argv[i + j]);
        const bool rows16 = fattn::mask_rows16((const void*)a[1], 0, 0, a[3], 1);
        printf("%d ", (int)fattn::mask_bits_pay(a[0], rows16, a[2], a[3], (int)a[4], (int)a[5], a[6]));
    }
}
"""


def test_rule(tmp_path):
    src, exe = tmp_path / "route.cpp", tmp_path / "route"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    at, off = 4096, 4097                       # a mask's address, on 16 bytes and not
    # backward, address, a mask for every head, row stride, Sq, Sk, causal, (unused) -> bits
    cases = [((0, at, 0, 1216, 1216, 1216, 0, 0), 1), ((0, at, 0, 1152, 1152, 1152, 0, 0), 0), ((0, at, 1, 2048, 2048, 2048, 0, 0), 0),
             ((0, off, 1, 2048, 2048, 2048, 0, 0), 1), ((0, at, 1, 2000, 2000, 2000, 0, 0), 1),
             ((1, at, 0, 1024, 1024, 1024, 0, 0), 1), ((1, at, 1, 1024, 1024, 1024, 0, 0), 1), ((1, at, 0, 896, 896, 896, 0, 0), 0),
             ((1, at, 0, 896, 896, 896, 1, 0), 1), ((1, at, 0, 832, 832, 832, 0, 0), 1), ((1, at, 0, 896, 900, 896, 0, 0), 1),
             ((1, at, 0, 896, 300, 896, 0, 0), 1), ((0, at, 0, 896, 300, 896, 0, 0), 0),
             ((1, at, 0, 1 << 26, 896, 896, 0, 0), 1), ((0, at, 0, 1024, 1024, 1024, 1, 0), 1), ((0, at, 0, 896, 896, 896, 1, 0), 0), ((0, off, 0, 384, 384, 384, 0, 0), 1), ((0, off, 0, 256, 384, 256, 0, 0), 0),
             ((1, off, 0, 1, 1, 1152, 0, 0), 1), ((1, off, 0, 1, 1, 1088, 0, 0), 1), ((1, off, 0, 1, 1, 1024, 0, 0), 0)]
    out = subprocess.run([str(exe), *(str(x) for c, _ in cases for x in c)], check=True, capture_output=True, text=True).stdout.split()
    assert [int(x) for x in out] == [w for _, w in cases]
