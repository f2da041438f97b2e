"""Division by a number known beforehand (csrc/fast_div.hpp), compiled for the host: exact below 2^31 around every multiple tried."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include "fast_div.hpp"
int main() {
    uint64_t x = 88172645463325252ull;
    const uint32_t edge[] = {1, 2, 3, 5, 6, 7, 12, 16, 24, 77, 127, 128, 129, 1000, 4608, 65535, 65536, 1u << 30, (1u << 30) + 1, 0x7fffffffu};
    for (int i = 0; i < 3000; ++i) {
        x ^= x << 13; x ^= x >> 7; x ^= x << 17;
        const uint32_t d = i < 20 ? edge[i] : (uint32_t)(x >> (33 + x % 30)) + 1u;
        if (d > 0x7fffffffu) continue;
        const fattn::FastDiv f(d);
        for (int j = 0; j < 400; ++j) {
            x ^= x << 13; x ^= x >> 7; x ^= x << 17;
            uint64_t u = j < 4 ? 0x7fffffffull - j : j < 8 ? j - 4 : x >> 33;
            if (j & 1) u = u / d * d;
            if (j % 3 == 2 && u) --u;
            if (u > 0x7fffffffull || f((uint32_t)u) == u / d) continue;
            printf("%u / %u\n", (uint32_t)u, d);
            return 1;
        }
    }
    return 0;
}
"""


def test_exact(tmp_path):
    src, exe = tmp_path / "div.cpp", tmp_path / "div"
    src.write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
