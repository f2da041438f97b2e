"""Which unit a workgroup takes (csrc/xcd_order.hpp), compiled for the host: every unit once, contiguous ranges per XCD, and with
batches of unequal length the same share of every batch per XCD."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "xcd_order.hpp"
int unit(int linear, int total, int tiles, int B, int H, bool falling, bool by_batch, bool snake) {
    if (fattn::deals_units(total, tiles, B, H, falling, by_batch, 1)) {
        int tile, bh;
        if (snake) fattn::dealt_unit<true>(linear, tiles, B, H, by_batch, tile, bh);
        else fattn::dealt_unit<false>(linear, tiles, B, H, by_batch, tile, bh);
        return bh * tiles + tile;
    }
    if (by_batch) return snake ? fattn::xcd_remap_heads<true>(linear, total, tiles) : fattn::xcd_remap_heads<false>(linear, total, tiles);
    return fattn::xcd_remap(linear, total);
}
int main(int, char** argv) {
    const int B = atoi(argv[1]), H = atoi(argv[2]), tiles = atoi(argv[3]), total = B * H * tiles;
    for (int i = 0; i < total; ++i)
        printf("%d %d %d %d %d %d %d %d %d %d\n", unit(i, total, tiles, B, H, false, false, false), unit(i, total, tiles, B, H, true, false, false),
               unit(i, total, tiles, B, H, true, false, true), unit(i, total, tiles, B, H, false, true, false), unit(i, total, tiles, B, H, false, true, true),
               fattn::xcd_remap_split(i, total), fattn::xcd_remap_tiles(i, total, tiles, false), fattn::xcd_remap_tiles(i, total, tiles, true),
               fattn::xcd_remap_heads(i, total, tiles, false, false), fattn::xcd_remap_heads(i, total, tiles, false, true));
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "flame_amd", "csrc"), str(d / "order.cpp"), "-o", str(d / "order")], check=True)
    return str(d / "order")


@pytest.mark.parametrize("batches,heads,tiles", [(1, 1, 1), (1, 1, 9), (3, 1, 300), (1, 7, 1), (2, 8, 4), (1, 9, 1), (3, 12, 9), (3, 30, 9), (9, 4, 17), (4, 16, 9),
                                                 (5, 15, 13), (13, 10, 5), (143, 7, 3), (2, 12, 40), (1, 1, 625), (1, 1, 961)])
def test_every_unit_once(exe, batches, heads, tiles):
    out = subprocess.run([exe, str(batches), str(heads), str(tiles)], check=True, capture_output=True, text=True).stdout.split()
    plain, falling, falling_snake, by_batch, by_batch_snake, split, even_tiles, causal_tiles, no_heads, no_heads_in_turn = ([int(v) for v in out[i::10]] for i in range(10))
    total = batches * heads * tiles
    for ids in (plain, falling, falling_snake, by_batch, by_batch_snake):
        assert sorted(ids) == list(range(total))
    assert split == (plain if total % 8 == 0 else list(range(total)))      # the workgroups that share walks: in turn where eight does not divide
    assert no_heads == plain and no_heads_in_turn == split
    assert causal_tiles == split and even_tiles == (split if total == tiles and total <= 768 else plain)         # score tiles of wide heads
    for x in range(8):
        mine = plain[x::8]
        assert mine == list(range(mine[0], mine[0] + len(mine))) if mine else True
    if heads % 8 != 0 and total > 256:            # every XCD has its eighth of every batch, but for the tiles dealt one by one
        for ids in (by_batch, by_batch_snake):
            for b in range(batches):
                share = [sum(v // tiles // heads == b for v in ids[x::8]) for x in range(8)]
                assert max(share) - min(share) <= 1
        for x in range(8):                        # in the order of the batches, within the eight units dealt at a time
            seq = [v // tiles // heads for v in by_batch[x::8]]
            assert all(seq[i] <= seq[i + heads] for i in range(len(seq) - heads))


# Score tiles of wide heads under the causal flag, in bands of eight key tiles with the query tiles across: the XCDs' shares of those that are attended to differ by
# no more than a band's eight columns do.  (In contiguous ranges an XCD has 0 to 28 of 15 x 15, 6 to 78 of 25 x 25, 15 to 120 of 31 x 31.)
@pytest.mark.parametrize("side", [15, 25, 31])
def test_causal_tiles_are_shared_out(exe, side):
    out = subprocess.run([exe, "1", "1", str(side * side)], check=True, capture_output=True, text=True).stdout.split()

    def attended(wg):
        band, j = divmod(wg, 8 * side)
        width = min(8, side - 8 * band)
        return 8 * band + j % width <= j // width

    share = [sum(attended(int(v)) for v in out[7::10][x::8]) for x in range(8)]
    assert sum(share) == side * (side + 1) // 2 and max(share) - min(share) <= 8 * ((side + 7) // 8), share
