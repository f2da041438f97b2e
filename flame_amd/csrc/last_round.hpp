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

}  // namespace fattn
