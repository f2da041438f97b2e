// 256-query workgroups, one per compute unit, which read K and V half as often, or 128-query ones, two of which share a unit: the
// rules of the forward, dQ and the Sage forward.  Host arithmetic only, so that it can be checked without a GPU.
//
// The 256-query kernels need more time from launch to first step and from last step to result (the forward's 64-query wavefronts
// 16 us, their first pass through 40 KB of code among it, its 128-query ones 10), a second 128-query workgroup on the unit covers the
// start and the end of the first, and twice as many of half the size fill a last round more evenly.  Against that stands a step that
// is cheaper by a few percent, less at D = 64 than at 128.  So 128-query workgroups serve short walks, last rounds that are at
// most half full, and walks of unequal length.
// `total`: the problem's 256-query workgroups, `cus`: compute units.  Figures: microseconds with 256- -> 128-query workgroups,
// total / cus in brackets, all inputs in place and the same.
#pragma once
#include "last_round.hpp"

namespace fattn {

// Under the causal flag: the second round is (nearly) full, so that every unit gets one of the longest walks and then one of the
// shortest.  From 6144 queries on it may lack a little more.
inline bool second_round_levels(int64_t total, int64_t cus, int N_q) {
    return 16 * total > (N_q > 6144 ? 27 : 29) * cus && total <= 2 * cus;
}

// Forward.  Nothing is excluded at all (plain) or the last key tile is cut, the causal flag is set, or there are key lengths, which keep
// 256-query workgroups wherever a last round allows it.  DP: padded head dim, d96: the kernels of 96.  These, and causal calls
// with another number of keys than queries, were not measured on both sides: their lines are those of last_round.hpp alone.
//
// Plain, D = 128: 512 keys [1.12] 35.2 -> 32.4, [1.5] 43.2 -> 35.8, [2] 50.4 -> 45.0, [4] 96.5 -> 85.0; 768 keys [1.12] 43.0 -> 41.6; 1024 keys [1.06] 48.8 ->
// 51.2, [1.12] 50.8 -> 51.8, [1.5] 61.2 -> 55.7, [2.25] 96.5 -> 85.1; 2048 keys [1.5] 101.2 -> 99.4, [1.75] 113.5 -> 119.9, [2.5] 164.8 -> 158.9; 3072 keys
// [1.5] 142.1 -> 143.2.  D = 64: 512 keys [1.12] 21.3 -> 20.0, [4] 57.1 -> 51.1; 768 keys [1.12] 26.3 -> 26.2; 1024 keys [1.06] 30.9 -> 32.0, [1.12] 31.3 ->
// 32.3, [1.5] 40.2 -> 35.2, [4] 91.1 -> 85.2; 1536 keys [1.12] 40.5 -> 44.5; 3072 keys [1.5] 90.0 -> 87.7, [1.75] 106.2 -> 107.2; 4096 keys [1.5] 116.3 -> 114.2.
// (On an eighth of the units a last round is cut into 32-query workgroups, launch_fwd_wide: hence the lower line there.)
// The last tile cut, D = 128: 499 keys [1.12] 36.0 -> 30.9, [2] 43.8 -> 42.2, [3] 66.9 -> 62.2; 1011 keys [1.5] 59.2 -> 54.0, [2] 69.1 -> 69.5, [2.5] 93.6 -> 85.9;
// 2035 keys [1.12] 105.0 -> 91.2, [1.5] 106.5 -> 98.3, [1.75] 112.1 -> 119.0, [2.5] 166.8 -> 158.3, [3] 183.2 -> 187.5.
// Causal, D = 128, as many keys as queries: 1024 [1] 30.5 -> 26.0, [2] 49.8 -> 48.5; 1536 [1] 42.3 -> 34.8, [1.88] 58.5 -> 59.9, [3] 103.3 -> 92.7; 2048 [1] 51.4 ->
// 43.0, [1.5] 58.7 -> 59.1, [2] 74.6 -> 76.2, [3] 123.9 -> 116.5; 3072 [1.5] 83.9 -> 80.9, [1.88] 97.9 -> 102.6, [3] 159.3 -> 151.9, [6] 333.7 -> 314.5; 4096 [1] 94.6 ->
// 78.8, [2] 129.4 -> 136.7; 8192 [1] 179.5 -> 147.6, [2] 241.9 -> 259.3, [4] 474.8 -> 480.8; slices that do not divide by the eight XCDs, which come in the order
// of causal_order.hpp: 1536 [1.99] 67.1 -> 62.4, 4096 [1.75] 126.3 -> 124.5, 6144 [1.97] 195.0 -> 197.6, 8192 [1.5] 207.0 -> 195.7, [1.75] 222.4 -> 232.0, [2.5] 326.0 -> 309.5,
// 16384 [1.75] 433.7 -> 455.6.
inline bool fwd_takes_256(int64_t total, int64_t cus, int64_t slices, int N_q, int N_kv, int DP, bool d96, bool causal, bool kv_len) {
    const bool plain = !causal && !kv_len && N_kv % 64 == 0, d64 = DP == 64;
    if (!plain && d64) return false;
    const bool eighth = thin_last_round(total, cus, 8), half = thin_last_round(total, cus, 2);
    if (!d96 && !kv_len && !causal && total > cus && !(plain && thin_last_round(total, cus, 32))) {     // (a handful more than whole rounds are cut cheaply)
        const int short_walk = plain && eighth ? (total < 2 * cus ? 768 : 1024) : half ? (d64 ? 3072 : 2048) : d64 ? 1024 : 512;
        if (N_kv <= short_walk) return false;
    }
    if (!d96 && !kv_len && causal && N_q > 768 && N_kv == N_q && !(second_round_levels(total, cus, N_q) && N_q >= (slices % 8 == 0 ? 1536 : 6144)) &&
        (N_kv <= 3072 || total <= cus || slices % 8 != 0))
        return false;
    return !thin_last_round(total, cus, 3) || (plain && (total >= 2 * cus || eighth));
}

// dQ; D: the kernels' head dim.  With key lengths or the causal flag the longest walks set the time, and the last round cannot be cut.
// Backward, all walks equally long, D = 128: 512 keys [1] 75.0 -> 73.4, [2] 148.2 -> 135.9, [4] 335 -> 301; 1024 keys [1] 115.8 -> 117.4, [2] 230.7 -> 224.1, [4] 513 -> 478;
// 1536 keys [2] 316.3 -> 313.0, [2.5] 421.5 -> 420.2, [4] 693 -> 653; 2048 keys [2.5] 517 -> 501, [2.75] 570.5 -> 571.8, [4] 815 -> 803; 3072 keys [3] 857 -> 868.
// D = 64: 512 keys [2] 76.5 -> 69.9, [4] 150.7 -> 130.5; 1024 keys [2] 123.9 -> 120.1, [4] 242.4 -> 230.6; 2048 keys [2] 221.3 -> 222.0, [2.5] 282.2 -> 275.0, [3] 328.1 -> 326.5,
// [4] 437.0 -> 431.6; 3072 keys [2.5] 403.0 -> 399.1, [2.75] 451.6 -> 458.0, [3] 473.8 -> 478.0; 4096 keys [2.5] 526.7 -> 527.5, [3] 614.9 -> 629.1.
// Causal, as many keys as queries, D = 128: 1024 [1] 103.4 -> 90.5, [2] 177.7 -> 165.3; 2048 [1] 159.7 -> 143.0, [4] 585 -> 536; 3072 [1.88] 332.9 -> 331.5, [3] 529 -> 505, [4.12] 784 ->
// 728; 4096 [1] 252.4 -> 228.5, [2] 424.0 -> 431.8; 8192 [2] 774 -> 806, [3] 1177 -> 1179; D = 64: 1024 [1] 60.1 -> 50.0, [2] 101.7 -> 89.2; 2048 [2] 153.8 -> 148.0, [4] 294.3 -> 269.2;
// 4096 [1] 174.0 -> 155.8, [2] 246.1 -> 246.4, [4] 492 -> 476; 8192 [1.75] 401.9 -> 408.5, [2] 448 -> 459, [4] 884.1 -> 886.4.
inline bool dq_takes_256(int64_t total, int64_t cus, int N_q, int N_kv, int D, bool causal, bool kv_len) {
    const bool even = !causal && !kv_len, half = thin_last_round(total, cus, 2);
    if (half && (!even || total < 2 * cus)) return false;
    if (N_kv <= 1024 && (even ? total > cus : total % cus != 0)) return false;
    if (D == 96) return true;
    if (causal && !kv_len && N_q > 768 && N_kv == N_q && (N_kv <= (D == 64 ? 4096 : 3072) || total <= cus)) return false;
    return !(even && 4 * total >= 9 * cus && N_kv <= (D == 64 ? (half ? 3072 : 2048) : 1536));
}

// Sage forward, without exclusions.  A last round on at most half of the units is cut into 128-query workgroups in a launch of its own: up to
// 1024 keys the start of that costs more than it gains.  (Cut -> 128-query workgroups throughout, D = 128: 512 keys [1.12] 34.1 -> 30.3, [1.5] 35.4 ->
// 30.4, [2.5] 54.5 -> 46.7; 1024 keys [1.12] 49.8 -> 46.9, [2.5] 79.8 -> 76.0; 1536 keys [1.5] 68.0 -> 66.6, [2.5] 107.4 -> 120.6; 2048 keys [1.5] 84.9 -> 85.3; D = 64: 512 keys [1.25]
// 23.9 -> 22.6; 1024 keys [1.12] 35.1 -> 33.0, [2.5] 54.7 -> 51.3; 1536 keys [1.5] 46.8 -> 44.8, [2.5] 76.7 -> 81.7.)
inline bool sage_takes_256(int64_t total, int64_t cus, int N_kv) { return !(total > cus && thin_last_round(total, cus, 2) && N_kv <= 1024); }

}  // namespace fattn
