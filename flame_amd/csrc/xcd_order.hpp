// Which unit of a problem a workgroup takes, so that the units that read the same keys and values share an XCD's L2: integer
// arithmetic only, so that it can be checked without a GPU.
#pragma once
#include "causal_order.hpp"

namespace fattn {

// Workgroups are dealt to the 8 XCDs (each with its own L2) round-robin by linear id.  Remap the id
// so that XCD x works on the contiguous range [x*total/8, (x+1)*total/8) of tiles: all tiles of one
// (batch, head) then share one L2 and its K/V (forward) or Q/dO (backward) stay resident there.
// Where the total does not divide, the first total % 8 ranges are one longer, as the shares of the XCDs are.
FATTN_HOST_DEVICE int xcd_remap(int linear, int total) {
    constexpr unsigned kXcd = 8;
    const unsigned l = (unsigned)linear, t = (unsigned)total, x = l % kXcd;
    return (int)(x * (t / kXcd) + (x < t % kXcd ? x : t % kXcd) + l / kXcd);
}
// Workgroups that share one walk: in turn where the total does not divide.  (Contiguous ranges there, dK/dV, us: 7 heads of 1500 D=64, 252 workgroups,
// 16.6 -> 21.0, D=128 25.1 -> 27.7; 5 heads of 1100 D=96, 180 workgroups, 17.2 -> 19.5.  dQ 1 to 3 % at D=64 and 96.)
FATTN_HOST_DEVICE int xcd_remap_split(int linear, int total, bool in_turn = true) { return in_turn && total % 8 != 0 ? linear : xcd_remap(linear, total); }
// The same for P V of wide heads.  (Contiguous ranges there, us: one head of D = 512, S = 1200 19.2 -> 19.8, 2300 19.3 -> 19.9, 3200 24.9 -> 27.0; three heads of
// D = 320, S = 2300 35.4 -> 37.7, causal 33.0 -> 32.1, S = 3968 75.5 -> 74.0, causal 54.7 -> 56.7.)
// Tiles of the scores of wide heads: in turn under the causal flag, as ever fewer tiles of the later bands of keys are attended to and contiguous
// ranges are unequal shares, and on small grids of one slice, whose rows all L2s hold; 768: one and a half rounds of two workgroups per compute unit.  (In
// turn -> contiguous, us, scores of the backward / probabilities of the forward: causal, one head of D = 512, S = 1800 17.9 -> 19.0 / 11.8 -> 13.2, S = 3200
// 23.6 -> 36.0 / 14.7 -> 21.9, S = 3968 36.4 -> 42.8 / 22.7 -> 25.9, three of D = 320, S = 3968 60.7 -> 68.0 / 36.2 -> 42.7; without it 100 tiles 18.2 -> 18.9 / 13.7 ->
// 13.6, 225 19.2 -> 19.5 / 12.7 -> 14.5, 324 23.9 -> 24.4 / 14.7 -> 15.6, 625 38.5 -> 39.0 / 22.9 -> 23.1, 961 53.9 -> 49.9 / 33.0 -> 29.4, 972 39.3 -> 40.7 / 25.0 -> 24.6, 2883
// 112.7 -> 98.1 / 61.3 -> 59.0.  Of several slices an XCD
// keeps its own: four of 81 tiles, D = 264 21.0 -> 19.4 / 13.7 -> 12.9, three of 100 23.5 -> 23.2 / 15.3 -> 15.3.  The products of the backward gain by contiguous ranges, 300 workgroups 53.2 -> 45.6, 837 160 -> 128, causal 120 -> 80.)
FATTN_HOST_DEVICE int xcd_remap_tiles(int linear, int total, int per_slice, bool causal) {
    return xcd_remap_split(linear, total, causal || (per_slice == total && total <= 768));
}
// Workgroups of which a compute unit holds two are dealt out one per unit, then a second one each.  Where (nearly) all fit at once
// nothing is left to even out unequal walks: in the order of falling length the units with the longest walks would get the
// longer ones of the second deal as well, so that one is turned round.  With more than three deals the order of falling length
// is better: the units that finish first take what is left.
// (Forward and backward, us: B=4 H=16 S=1101 D=128 key mask 154.5 -> 150.7, B=4 H=16 1024 x 2049 D=64 key lengths 123.5 -> 121.5,
// B=1 H=16 S=3000 D=128 causal 203 -> 198, its forward 55.3 -> 52.7; four deals turned in pairs: B=4 H=32 S=1024 D=64 causal,
// forward 27.8 -> 29.2.)
// j: place in the order of the `total` workgroups of an XCD with 32 compute units (the whole card's; with another number the
// order is another one, as complete).
FATTN_HOST_DEVICE int snake_order(int j, int total) {
    constexpr int kUnits = 32;
    const int end = total < 2 * kUnits ? total : 2 * kUnits;
    return total <= 3 * kUnits && j >= kUnits && j < end ? kUnits + end - 1 - j : j;
}
// The same for batches whose sequences differ in length (per-batch key lengths): contiguous ranges would hand
// whole batches, the long ones and the short ones, to different XCDs.  Here XCD x takes the (batch, head)
// slices x, x + 8, x + 16, ...: every slice still stays in one L2, and the heads of one batch are spread
// over all XCDs.  `per_head`: tiles per (batch, head) slice; the id runs slice-major.
// SNAKE: workgroups of which a compute unit holds two, the longest walks first: see snake_order.
// by_heads: whether this order is wanted at all; in_turn: else, whether a total that does not divide goes in turn (under the causal flag all
// workgroups are in one order then, from the longest walk to the shortest: causal_longest_first).  One call for all three orders, whose result alone is
// divided: 40 to 60 instructions fewer ahead of a kernel's first load than with the choice in every kernel and a second division under the causal flag.
// (Forward, us: 4 x 8 heads of 257, D = 72 8.64 -> 8.40, D = 128 9.85 -> 9.62, 2 x 16 of 577, D = 64 10.08 -> 9.86; forward and backward with dropout, B=2 H=16 S=1024
// D=64 63.98 -> 63.31.)
template <bool SNAKE = false>
FATTN_HOST_DEVICE int xcd_remap_heads(int linear, int total, int per_head, bool by_heads = true, bool in_turn = true) {
    constexpr int kXcd = 8;
    if (!by_heads || total / per_head % kXcd != 0) return xcd_remap_split(linear, total, by_heads || in_turn);
    const int x = linear % kXcd, j = SNAKE ? snake_order(linear / kXcd, total / kXcd) : linear / kXcd;
    return ((j / per_head) * kXcd + x) * per_head + j % per_head;
}

// Problems whose walks differ in length and whose slices do not divide by the XCDs: the units left over are dealt one by one
// (causal_order.hpp).  Under the causal flag (falling): all B H slices, `tile` counted from the longest walk.  Where the batches differ
// (by_batch: key lengths or key masks of several batches, masks as bits): the H heads of every batch, batch after batch, wherever H does not divide,
// also where B H does and every XCD could keep whole slices: it would get long ones or short ones.  (That order -> this one, mean over 8 draws of key
// lengths, forward / dK/dV / dQ, 4096 x 4096, D = 128: B=4 H=4 1.08 / 1.14 / 1.08 times as fast, B=8 H=4 1.06 / 1.10 / 0.99, B=8 H=2 1.13 / 1.13 / 1.15, B=8 H=12
// 1.02 / 1.06 / 1.05; B=8 H=4 at D = 64 1.09 / 1.09 / 1.00.  One batch has nothing to level: B=1 H=12 4096 x 4096 D=128 with a key mask, backward 349 -> 353 us.)
// deals_units: the host's choice between a kernel's two instances.  (As a condition within the kernels it was 200 to 270 instructions ahead of every
// problem's first load: forward, us, B=4 H=16 S=1101 D=128 with a key mask 40.2 -> 40.6, B=4 H=16 S=1101 D=64 30.5 -> 30.8.)
// least: the fewest tiles per slice under the causal flag.  (Forward with fewer than eight: 75 heads of 512 at D = 64 11.0 -> 12.1 us, 107 of 1024 with
// 256-query workgroups 46.8 -> 53.4.)
inline bool deals_units(int64_t total, int tiles, int B, int H, bool falling, bool by_batch, int least) {
    return (by_batch || (falling && tiles >= least)) && causal_order_pays(by_batch ? H : (int64_t)B * H, total);
}
template <bool SNAKE = false>
FATTN_HOST_DEVICE void dealt_unit(int linear, int tiles, int B, int H, bool by_batch, int& tile, int& bh) {
    int slice, level;
    causal_order(linear, by_batch ? H : B * H, by_batch ? B * tiles : tiles, slice, level, [](int j, int count) { return SNAKE ? snake_order(j, count) : j; });
    tile = by_batch ? level % tiles : level;
    bh = by_batch ? level / tiles * H + slice : slice;
}

}  // namespace fattn
