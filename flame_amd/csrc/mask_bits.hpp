// A keep-mask that differs by query, as bits: one pass over its bytes leaves, per 64 x 64 tile of (query, key), a 64-bit word of
// keys for every query, a word of queries for every key, and a flag that says whether anything of the tile is attended and
// whether all of it is.  The attention kernels then walk the attended tiles only, those attended whole without a test per
// element, and a lane whose query (forward, dQ) or key (dK/dV) meets a cut tile loads one word for it, 8 bytes next to its
// neighbours', instead of 64 bytes of a row of its own.  Key lengths and the causal flag are folded in.
// Packed sequences, which attend to themselves, are the case it is made for: B=2 H=16 S=1500, four documents each, D = 64 forward
// 221 -> 34 us and backward 832 -> 78, D = 128 543 -> 51 and 967 -> 153 us, of which the pass over the mask takes 4 us twice.  Where
// every tile is cut (each element of a mask kept by chance) the words cost about what the rows did where those could be loaded
// in vectors: B=2 H=16 S=1536 D = 128 62 -> 64 and 174 -> 170 us, with S=1500 543 -> 57 and 968 -> 168 us.
// The kernels that read the mask itself serve the call where the bits would not pay (mask_route.hpp) and where there is no room for
// the words (flame_attn_mask_workspace_bytes).
#pragma once
#include "attn_common.hpp"

namespace fattn {

struct MaskBitsParams {
    MaskArgs m;
    int Sq, Sk, H;                // H: heads per batch among the planes (1 where all heads share one)
    int n_qt, n_kt;               // tiles of 64, padded to even numbers
    uint64_t *rows, *cols;
    uint8_t* flags;
};

// The 64 x 64 bits that lane k holds row k of, transposed: lane k gets column k.
__device__ __forceinline__ uint64_t transpose_bits64(uint64_t x) {
    const int lane = threadIdx.x & 63;
    static_for<6>([&](auto i_tag) {
        constexpr int i = decltype(i_tag)::value, j = 32 >> i;
        // blocks of j rows and columns: the upper right one changes places with the lower left one
        constexpr uint64_t low = j == 32 ? 0x00000000ffffffffull : j == 16 ? 0x0000ffff0000ffffull : j == 8 ? 0x00ff00ff00ff00ffull
                               : j == 4 ? 0x0f0f0f0f0f0f0f0full : j == 2 ? 0x3333333333333333ull : 0x5555555555555555ull;
        const uint64_t y = ((uint64_t)(uint32_t)__shfl_xor((int)(x >> 32), j, 64) << 32) | (uint32_t)__shfl_xor((int)x, j, 64);
        x = lane & j ? (x & ~low) | ((y >> j) & low) : (x & low) | ((y & low) << j);
    });
    return x;
}
// one bit per byte that is not zero, of sixteen
__device__ __forceinline__ uint32_t nonzero_bytes16(u32x4 w) {
    uint32_t out = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t high = ((w[i] | ((w[i] & 0x7f7f7f7fu) + 0x7f7f7f7fu)) & 0x80808080u) >> 7;
        out |= ((high * 0x01020408u) >> 24 & 0xfu) << (4 * i);
    }
    return out;
}

// One wavefront per tile.  ROWS: uint8, at least 16 keys, contiguous along them: four lanes load the 64 bytes of a row, whatever its
// alignment (one that would reach past the row's end loads its last 16 bytes), and their bits meet in LDS as its word: one plane
// of 1500 x 1500 3.6 us.  Otherwise lane = key, and a row's word is the ballot of 64 loads: 15.3 us.
template <bool ROWS>
static __global__ __launch_bounds__(256) void mask_bits_kernel(const MaskBitsParams p) {
    __shared__ alignas(8) uint16_t pieces[4][64 * 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_plane = p.n_qt * ((p.n_kt + 3) / 4);
    const int plane = blockIdx.x / per_plane, at = blockIdx.x % per_plane;
    const int u = at % p.n_qt, t = at / p.n_qt * 4 + wave;
    if (t >= p.n_kt) return;
    const int b = plane / p.H, hh = plane % p.H;
    const uint8_t* base = mask_head_base(p.m, b, hh);
    int klimit = p.Sk;
    if (p.m.kv_len) klimit = min(klimit, max(p.m.kv_len[b], 0));
    const int key = 64 * t + lane, n_rows = min(64, p.Sq - 64 * u), n_keys = min(64, klimit - 64 * t);      // may be negative: padding
    const uint64_t keys_ok = n_keys >= 64 ? ~0ull : n_keys <= 0 ? 0ull : (1ull << n_keys) - 1;
    uint64_t row = 0;                                  // of query 64 u + lane
    if constexpr (ROWS) {
        typedef u32x4 __attribute__((aligned(1))) piece_t;
        const int k = 64 * t + 16 * (lane & 3), k_at = min(k, p.Sk - 16);
        u32x4 w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * i + (lane >> 2);
            w[i] = u32x4{0u, 0u, 0u, 0u};
            if (r < n_rows && k < p.Sk) w[i] = *reinterpret_cast<const piece_t*>(base + (int64_t)(64 * u + r) * p.m.sq + k_at);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) pieces[wave][64 * i + lane] = (uint16_t)(nonzero_bytes16(w[i]) >> min(k - k_at, 16));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");                 // the wavefront's own LDS operations, in their order
        __builtin_memcpy(&row, __builtin_assume_aligned(&pieces[wave][4 * lane], 8), 8);
    } else {
#pragma unroll 32
        for (int r = 0; r < 64; ++r) {
            const int q = 64 * u + r;
            const uint64_t w = __ballot(key < p.Sk && r < n_rows &&
                                        mask_attends(p.m, base, (int64_t)min(q, p.Sq - 1) * p.m.sq + (int64_t)min(key, p.Sk - 1) * p.m.sk));
            row = lane == r ? w : row;
        }
    }
    row &= keys_ok;
    if (p.m.causal) {
        const int n = 64 * u + lane - 64 * t + 1;      // keys up to the query
        row &= n >= 64 ? ~0ull : n <= 0 ? 0ull : (1ull << n) - 1;
    }
    if (lane >= n_rows) row = 0;
    const uint64_t col = transpose_bits64(row);
    p.rows[((int64_t)plane * p.n_kt + t) * (64 * p.n_qt) + 64 * u + lane] = row;
    p.cols[((int64_t)plane * p.n_qt + u) * (64 * p.n_kt) + key] = col;
    const bool any = __any(row != 0);
    const bool all_keys = __all(lane >= n_rows || row == ~0ull);              // every query that exists attends to all 64 keys
    const bool all_rows = n_rows >= 64 && __all(row == keys_ok);              // 64 queries, and all attend to every key within the length
    if (lane == 0) p.flags[((int64_t)plane * p.n_qt + u) * p.n_kt + t] = (any ? kTileAny : 0) | (all_keys ? kTileAllKeys : 0) | (all_rows ? kTileAllRows : 0);
}

}  // namespace fattn
