// The order in which the workgroups of a causal problem start where its (batch, head) slices do not divide by the eight XCDs:
// integer arithmetic only, so that it can be checked without a GPU.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define FATTN_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define FATTN_HOST_DEVICE inline
#endif

namespace fattn {

// Up to one workgroup per compute unit the order is nothing but its divisions' time (0.3 us); the products below stay under 2^31.
inline bool causal_order_pays(int64_t slices, int64_t total) { return slices % 8 != 0 && total > 256 && total <= 1 << 18; }

// Workgroup `linear` of `slices` * `levels`, slices % 8 != 0: its slice and its level, 0 being the longest walk of a slice.
// Workgroups go to the XCDs in turn by `linear`.  An XCD keeps floor(slices / 8) whole slices, whose K and V stay in its L2; the
// units of the up to seven slices left over are dealt to all eight, and every XCD takes its share of them spread evenly among
// its own, so that all of them walk from the longest to the shortest and end together.  (Contiguous eighths of the units give one
// XCD the long walks of a slice and the next one the short.  Forward, us, those -> this order: D = 128, 36 slices of 1024 29.2 -> 22.7, 30 of 2048
// 53.6 -> 42.4, 75 of 2048 125.5 -> 100.3, 12 of 4096 96.5 -> 73.6, 107 of 4096 496 -> 471; D = 64, 36 of 1024 20.3 -> 15.9, 30 of 3072 66.4 -> 49.0,
// 12 of 8192 156.6 -> 125.8.  Backward: D = 128, 36 of 1024 82.3 -> 60.2, 75 of 2048 325 -> 296, 12 of 8192 691 -> 622; D = 64, 43 of 3072 244 -> 188,
// 43 of 8192 1280 -> 1144.)
// place(j, count): where the XCD's j-th workgroup of `count` stands in that sequence.
template <class Place>
FATTN_HOST_DEVICE void causal_order(int linear, int slices, int levels, int& slice, int& level, Place&& place) {
    const int own = slices / 8, left = slices % 8, x = linear % 8;
    const int n_left = (left * levels - x + 7) / 8, count = own * levels + n_left;         // of this XCD
    const int j = place(linear / 8, count);
    const int before = j * n_left / count;                                                 // left-over units ahead of the j-th
    if ((j + 1) * n_left / count > before) {
        const int u = 8 * before + x;
        level = u / left;
        slice = 8 * own + u % left;
    } else {
        const int o = j - before;
        level = o / own;
        slice = o % own * 8 + x;
    }
}

}  // namespace fattn
