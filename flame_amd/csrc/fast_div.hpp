// Division of numbers below 2^31 by a number known before the launch: a multiplication and a shift (five vector instructions; the
// general 32-bit division takes about thirty).
#pragma once
#include <stdint.h>

namespace fattn {

// q = u m / 2^s with m = floor(2^s / d) + 1 and s = 31 + ceil(log2 d): m d exceeds 2^s by at most d <= 2^(s - 31), so that the
// quotient is too large by less than u / 2^31 / d < 1 / d: never enough to reach the next whole number.
struct FastDiv {
    uint32_t d, m, s;
    explicit FastDiv(uint32_t divisor) : d(divisor), s(31) {
        while (((uint64_t)1 << (s - 31)) < d) ++s;
        m = (uint32_t)(((uint64_t)1 << s) / d + 1);
    }
#if defined(__HIPCC__)
    __host__ __device__
#endif
    uint32_t operator()(uint32_t u) const { return (uint32_t)(((uint64_t)u * m) >> s); }
};

}  // namespace fattn
