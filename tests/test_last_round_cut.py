"""The arithmetic that cuts the last round of 256-query workgroups into smaller ones (csrc/last_round.hpp), on the CPU: over
query counts with every kind of last tile, numbers of (batch, head) slices and of compute units, the launches together take
every tile of 32 queries of the problem once and no id lies outside of it."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "last_round.hpp"
extern "C" void cut(int Sq, long slices, long cus, int share, long* out) {
    const fattn::LastRound r = fattn::cut_last_round(Sq, slices, cus, share != 0);
    out[0] = r.wide; out[1] = r.rows; out[2] = r.base; out[3] = r.count;
}
"""


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    d = tmp_path_factory.mktemp("last_round")
    (d / "cut.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-fPIC", "-shared", "-I" + os.path.join(ROOT, "flame_amd", "csrc"),
                    str(d / "cut.cpp"), "-o", str(d / "cut.so")], check=True)
    f = ctypes.CDLL(str(d / "cut.so")).cut
    f.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long, ctypes.c_int, ctypes.POINTER(ctypes.c_long)]

    def call(Sq, slices, cus, share):
        out = (ctypes.c_long * 4)()
        f(Sq, slices, cus, share, out)
        return tuple(out)
    return call


def _taken(Sq, slices, rows, first, count):
    """32-query tiles of the problem that workgroups first .. first + count - 1 of `rows` queries take, as the kernels read ids:
    tile id % n_qt of slice id // n_qt."""
    n_qt, n32 = -(-Sq // rows), -(-Sq // 32)
    for wg in range(first, first + count):
        s, q0 = wg // n_qt, wg % n_qt * rows
        assert s < slices, f"{Sq=} {slices=}: workgroup {wg} of {rows} queries lies past the problem"
        for t in range(q0 // 32, min((q0 + rows) // 32, n32)):
            yield s * n32 + t


def _check(Sq, slices, cus, share, got):
    wide, rows, base, count = got
    seen = list(_taken(Sq, slices, 256, 0, wide))
    if count:
        assert rows in ((32, 128) if share else (128,)) and (rows == 128 or count <= cus)
        seen += _taken(Sq, slices, rows, base, count)
    n = slices * -(-Sq // 32)
    assert len(seen) == n and len(set(seen)) == n, f"{Sq=} {slices=} {cus=} {share=}: {len(seen)} of {n} tiles, {len(set(seen))} different"


# whole wide tiles, odd and even counts of 128-query tiles, tiles of 32 left out of the last 128, ragged by one row
SIZES = sorted({256 * n - cut_off for n in (1, 2, 3, 6, 12, 17) for cut_off in (0, 1, 31, 32, 33, 64, 96, 127, 128, 129, 200, 255)})


@pytest.mark.parametrize("cus", [256, 304, 38, 7])
def test_every_tile_once(cut, cus):
    cuts = 0
    for Sq in SIZES:
        n = -(-Sq // 256)
        for slices in sorted({1, 2, 5, 16, 24, 48, 130, 180, (cus + 1) // n + 1, (cus + cus // 8) // n + 1, 2 * cus // n + 1}):
            for share in (0, 1):
                got = cut(Sq, slices, cus, share)
                _check(Sq, slices, cus, share, got)
                cuts += got[3] > 0
    assert cuts > 20


def test_drifting_ids_are_not_cut(cut):
    """More wide tiles than pairs of 128-query ones: 272, 288 and 288 units on 256 compute units stay one launch."""
    for Sq, slices in ((4224, 16), (2944, 24), (1408, 48)):
        assert cut(Sq, slices, 256, 1)[1:] == (0, 0, 0)
    # the check above does see such a cut: the second launch at twice the wide count
    with pytest.raises(AssertionError):
        _check(4224, 16, 256, 1, (256, 128, 512, 32))
    # whole pairs: 288 units become 256 wide ones and 256 of 32 queries, or 64 of 128 where the last tile is ragged by more
    assert cut(1536, 48, 256, 1) == (256, 32, 2048, 256)
    assert cut(1500, 48, 256, 1) == (256, 128, 512, 64)
    assert cut(1536, 48, 256, 0) == (256, 128, 512, 64)
