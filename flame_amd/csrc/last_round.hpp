// How a grid of 256-query workgroups ends (forward, dQ and Sage forward): host arithmetic only, so that it can be checked
// without a GPU.
#pragma once
#include <stdint.h>

namespace fattn {

// The first `wide` workgroups of 256 queries run as such.  The queries of the others, if any, go to a launch of its own of
// `count` workgroups of `rows` queries, whose ids start at `base`.
// Both kinds of workgroup number the query tiles slice by slice ((batch, head) slices of ceil(Sq / rows) tiles each), so id
// `base` is the tile at which the wide workgroups stop only if every slice is 256 / rows small tiles per wide one: where a
// slice's last wide tile is filled less than that (Sq = 4224: 17 wide tiles, 33 of 128 queries) the ids of the two kinds drift
// apart by a tile per slice, and the small launch would leave tiles out and take ids past the problem.
struct LastRound {
    int64_t wide;
    int rows = 0;               // 0: no second launch
    int64_t base = 0, count = 0;
};

// A last round that would leave at least half of the compute units idle is cut: into 32-query workgroups while these fit one per
// unit (`share`: the kernel has them), else into 128-query ones.
inline LastRound cut_last_round(int Sq, int64_t slices, int64_t cus, bool share) {
    const int64_t n_qt = ((int64_t)Sq + 255) / 256, total = n_qt * slices, rest = total % cus;
    const auto whole = [&](int rows) { return ((int64_t)Sq + rows - 1) / rows == 256 / rows * n_qt; };
    LastRound r{total};
    if (total <= cus || rest == 0 || 2 * rest > cus || !whole(128)) return r;
    r.rows = share && 8 * rest <= cus && whole(32) ? 32 : 128;
    r.wide = total - rest;
    r.base = r.wide * (256 / r.rows);
    r.count = rest * (256 / r.rows);
    return r;
}

// Whether 128-query workgroups, two per compute unit, finish sooner than `total` 256-query ones, one per unit: their last round
// is finer, and a second workgroup covers the start and the end of the first, while 256-query ones read K and V half as often.
// Measured at D = 64 and 128, times with 256-query -> 128-query workgroups (total / 256 compute units in brackets):
//   forward without exclusions   [1.12] 89.7 -> 91.0 with the cut into 32-query ones, [1.25] 64.3 -> 61.9, 41.9 -> 39.0, [1.5] 87 -> 90, [1.69] 240 -> 263 us
//   forward, ragged or causal    [1.12] 78 -> 69, [1.17] 133 -> 114, [1.25] 72 -> 63, [1.5] 49.0 -> 50.2,
//                                [1.69] 252 -> 262, [2.0] 135 -> 144 us; D = 64, whatever the rounds: 159 -> 129 [1.12], 94 -> 87 [2.0]
//   backward (dQ)                [1.12] 231 -> 223, 127 -> 119, [1.25] 200 -> 194, [1.5] 174 -> 167, 247 -> 243, [1.69] 729 -> 762 us;
//                                causal [1.12] 228 -> 216, [2.25] 238 -> 220, [1.88], 1000 keys 178 -> 165, [2.0] 426 -> 437 us
inline bool thin_last_round(int64_t total, int64_t cus, int64_t share) {          // the last round on at most 1 / share of the units
    const int64_t rest = total % cus;
    return rest != 0 && share * rest <= cus;
}

}  // namespace fattn
