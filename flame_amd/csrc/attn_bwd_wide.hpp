// Backward for head dims above 128 (any multiple of 8), without keep-mask or dropout.  At these head dims the accumulators
// of a fused backward do not fit a wavefront (dK^T and dV^T of 32 keys at D = 512 alone are 512 registers per lane), so
// P and dS are formed once and kept as bf16 for the duration of the call:
//   bwd_wide_rows     -delta = -rowsum(dO * O) and LSE * log2(e) of every query row
//   bwd_wide_scores   S^T = K Q^T and dP^T = V dO^T, 128 keys x 128 queries per workgroup, both contractions over the head
//                     dim in one loop; P = exp2(S c - lse2) and dS = P (dP - delta) from the accumulators, stored as bf16
//   bwd_wide_products dV^T = dO^T P, dK^T = scale Q^T dS and dQ^T = scale K^T dS^T in one grid, 128 x 128 output tiles
// so the fp32 scores never leave registers and nothing element-wise runs as a pass of its own.  P and dS of a (batch, head)
// are [Sq, Sk] padded to multiples of 128 (zero there), so that the products need no tests in their loops; the launcher
// takes as many (batch, head) slices at a time as the workspace holds.  Tiles that the causal flag excludes are neither
// formed nor read.
// Tiles of 128 rows x 64 (or 64 x 128) elements, 16 KiB each, are copied global -> LDS by LDS-DMA through a ring of five
// (WideRing): rows of a tile are whole 128-byte cache lines, and while one pair of tiles is multiplied the next pair and half
// of the one after are on their way.  Two workgroups per compute unit.  Bound by what the L2s deliver: at S = 4096
// the scores ask 650 MB of them and the products 900 MB, 14 TB/s; the matrix cores are busy a third of the time.
// B=1 H=1 S=4096 D=512: scores 47 us (0.74 PFLOP/s), products 63 us (0.82 PFLOP/s); 66 and 82 us with tiles 32 deep in two
// stages, whose 64-byte rows fetched every line twice, and stores straight from the accumulators; 246 us for the whole
// backward by library GEMMs and separate passes.  B=3 H=2 S=640 D=512, where the library's 15 calls kept the host busy,
// forward and backward: 615 -> 80 us.
#pragma once
#include "attn_common.hpp"

namespace fattn {

struct BwdWideParams {
    const uint16_t *q, *k, *v, *o, *dout;
    const float* lse;
    uint16_t *dq, *dk, *dv;
    float *ndelta, *lse2;         // [B*H, Sq]
    uint16_t *probs, *ds;         // [slices, sq_pad, sk_pad]
    Strides qs, ks, vs, os, dos, dqs, dks, dvs;
    int B, H, Sq, Sk, d;
    int sq_pad, sk_pad;           // multiples of 128
    int bh0;                      // first (batch, head) slice of this launch
    int n_slices;                 // ... and how many
    float scale;
    const int32_t* kv_len;
    int causal;
};

constexpr int kWideTile = 128, kWideStep = 64;

// one wavefront per query row
static __global__ __launch_bounds__(256) void bwd_wide_rows_kernel(const BwdWideParams p) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= (int64_t)p.B * p.H * p.Sq) return;
    const int bh = (int)(row / p.Sq), qi = (int)(row % p.Sq);
    const int b = bh / p.H, hh = bh % p.H;
    const uint16_t* ro = p.o + b * p.os.b + hh * p.os.h + (int64_t)qi * p.os.n;
    const uint16_t* rd = p.dout + b * p.dos.b + hh * p.dos.h + (int64_t)qi * p.dos.n;
    float acc = 0.f;
    for (int c = lane * 8; c < p.d; c += 512) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(ro + c), g = *reinterpret_cast<const u32x4*>(rd + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc += bf16_lo(a[i]) * bf16_lo(g[i]) + bf16_hi(a[i]) * bf16_hi(g[i]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) {
        const float l = p.lse[row];
        p.ndelta[row] = -acc;
        p.lse2[row] = (l == -INFINITY) ? INFINITY : l * kLog2e;
    }
}

// Five 16 KiB tiles ("units") in LDS, used in pairs: phase j multiplies units 2 j and 2 j + 1.  At its start unit 2 j + 2 may
// still be on its way; then units 2 j + 3 and 2 j + 4 are requested into the slots of the pair that phase j - 1 has read.
// Four 1 KiB copies per wavefront and unit, so that the count of outstanding copies says which units have landed.
struct WideRing {
    static constexpr int UNITS = 5, UNIT_ELEMS = kWideTile * kWideStep;
    static constexpr int LDS_BYTES = UNITS * UNIT_ELEMS * 2;
    int a = 0;                                             // slot of the first unit of the current phase
    __device__ __forceinline__ int slot(int i) const { return a + i < UNITS ? a + i : a + i - UNITS; }
    __device__ __forceinline__ void next() { a = slot(2); }
    // The pair of this phase has landed for every wavefront, and every wavefront has its fragments of the previous pair.
    // One statement, so that no access to LDS moves across it.
    __device__ __forceinline__ static void landed(bool last) {
        if (last) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
};

// Copies of a unit of 128 rows x 64 elements of the head dim: 16 of 8 rows x 128 bytes, four per wavefront; copy i: rows
// 8 (4 wave + i) + lane / 8.  The swizzle of copies 0 and 2, and of 1 and 3, is the same, so two lane offsets per tensor do
// where all 128 rows exist.
struct WideRows {
    int row0, gran0, gran1;
    uint32_t lds0;
    __device__ __forceinline__ explicit WideRows(const uint16_t* lds) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
        row0 = 32 * wave + (lane >> 3);
        gran0 = (lane & 7) ^ swz<64>(row0);
        gran1 = (lane & 7) ^ swz<64>(row0 + 8);
        lds0 = lds_addr(lds) + 4096u * (uint32_t)wave;
    }
    static_assert(swz<64>(0) == swz<64>(16) && swz<64>(8) == swz<64>(24) && swz<64>(7) == swz<64>(23), "the swizzle repeats every 16 rows");
    // copy i (0 .. 3) of elements [64 t, 64 t + 64) of the rows from base on, `rows` of which exist, d the head dim
    __device__ __forceinline__ void issue(const uint16_t* base, int64_t stride, int rows, int d, int t, int slot, int i) const {
        const uint32_t dst = lds0 + 2u * (uint32_t)(slot * WideRing::UNIT_ELEMS) + 1024u * (uint32_t)i;
        const uint16_t* src = base + kWideStep * t;
        const int g = i & 1 ? gran1 : gran0;
        if (kWideStep * (t + 1) <= d && rows >= kWideTile)
            dma16u(src + 8 * i * stride, 2u * (uint32_t)(row0 * (int)stride + 8 * g), dst);
        else                                               // rows past the end re-read the last one; granules past the head dim:
            dma16u(src, 2u * (uint32_t)(min(row0 + 8 * i, max(rows - 1, 0)) * (int)stride + (kWideStep * t + 8 * g < d ? 8 * g : 0)), dst);     // filler, zeroed in the fragments
    }
    __device__ __forceinline__ void issue(const uint16_t* base, int64_t stride, int rows, int d, int t, int slot) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) issue(base, stride, rows, d, t, slot, i);
    }
};

// One phase: the eight copies it requests, copy(i), then acc += A B^T over its unit pair, four chunks of 16 contraction elements;
// a(c, u) and b(c, u) read the fragments of chunk c.  (Copies spread out between the MFMAs, and fragments read a chunk ahead
// in an order fixed by hand, were slower, 80 -> 91 us for a forward: the requests have to leave early.)
template <class A, class B, class Copy>
__device__ __forceinline__ void wide_phase(f32x16 (&acc)[2][2], A&& a, B&& b, Copy&& copy) {
#pragma unroll
    for (int i = 0; i < 8; ++i) copy(i);
#pragma unroll
    for (int c = 0; c < kWideStep / 16; ++c) {
        bf16x8 af[2], bf[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            af[u] = a(c, u);
            bf[u] = b(c, u);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = mfma32(af[x], bf[y], acc[x][y]);
    }
}
// The last step of a contraction over the head dim where `rest` < 64 elements are left, from tiles of rows: fragments at row
// offsets fa / fb (row, granule 2 c + h: the chunk only flips bits 4 and 5 of the offset).
__device__ __forceinline__ void wide_multiply_tail(f32x16 (&acc)[2][2], const uint16_t* a, const uint16_t* b, const int (&fa)[2], const int (&fb)[2], int rest) {
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int c = 0; c < kWideStep / 16; ++c) {
        if (16 * c >= rest) break;
        bf16x8 af[2], bf[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            af[u] = *reinterpret_cast<const bf16x8*>(a + (fa[u] ^ (16 * c)));
            bf[u] = *reinterpret_cast<const bf16x8*>(b + (fb[u] ^ (16 * c)));
            if (16 * c + 8 * h >= rest) af[u] = bf[u] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});   // both: a filler must not meet a zero as an infinity
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = mfma32(af[x], bf[y], acc[x][y]);
    }
}

// ---- P and dS.  Units of contraction step t: 4 t = K, + 1 = Q, + 2 = V, + 3 = dO (rows of 64 elements).
static __global__ __launch_bounds__(256, 2) void bwd_wide_scores_kernel(const BwdWideParams p) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int wk = wave & 1, wq = wave >> 1;          // this wavefront's 64 keys and 64 queries of the tile

    // bands of eight key tiles, query tiles across: the 64 workgroups that an XCD runs at a time share 8 + 8 tiles of rows
    const int n_kt = p.sk_pad / kWideTile, n_qt = p.sq_pad / kWideTile;
    const int wg = xcd_remap_tiles(blockIdx.x, gridDim.x, n_kt * n_qt, p.causal);
    const int slice = wg / (n_kt * n_qt), in_slice = wg % (n_kt * n_qt);
    const int band = in_slice / (8 * n_qt), in_band = in_slice % (8 * n_qt), width = min(8, n_kt - 8 * band);
    const int kt = 8 * band + in_band % width, qt = in_band / width;
    const int bh = p.bh0 + slice, b = bh / p.H, hh = bh % p.H;
    const int k0 = kt * kWideTile, q0 = qt * kWideTile;
    if (p.causal && k0 > q0 + kWideTile - 1) return;       // nothing of this tile is attended, and nothing reads it
    int klimit = p.Sk;
    if (p.kv_len) klimit = min(klimit, max(p.kv_len[b], 0));

    const int k_last = p.Sk - 1, q_last = p.Sq - 1, k_rows = p.Sk - k0, q_rows = p.Sq - q0;
    const uint16_t* kbase = p.k + b * p.ks.b + hh * p.ks.h + (int64_t)min(k0, k_last) * p.ks.n;
    const uint16_t* vbase = p.v + b * p.vs.b + hh * p.vs.h + (int64_t)min(k0, k_last) * p.vs.n;
    const uint16_t* qbase = p.q + b * p.qs.b + hh * p.qs.h + (int64_t)min(q0, q_last) * p.qs.n;
    const uint16_t* gbase = p.dout + b * p.dos.b + hh * p.dos.h + (int64_t)min(q0, q_last) * p.dos.n;
    const WideRows copies(lds);
    int fk[2], fq[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int rk = 64 * wk + 32 * u + n, rq = 64 * wq + 32 * u + n;
        fk[u] = rk * kWideStep + 8 * (h ^ swz<64>(rk));
        fq[u] = rq * kWideStep + 8 * (h ^ swz<64>(rq));
    }

    float rows_nd[2], rows_l2[2];                          // requested before the walk, so that its end does not wait for them
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int qi = q0 + 64 * wq + 32 * qb + n;
        rows_nd[qb] = qi < p.Sq ? p.ndelta[(int64_t)bh * p.Sq + qi] : 0.f;
        rows_l2[qb] = qi < p.Sq ? p.lse2[(int64_t)bh * p.Sq + qi] : INFINITY;
    }

    f32x16 s[2][2], dp[2][2];                              // [key block][query block]
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][qb][r] = dp[kb][qb][r] = 0.f;

    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;

    const int n_steps = (p.d + kWideStep - 1) / kWideStep;
    WideRing ring;
    copies.issue(kbase, p.ks.n, k_rows, p.d, 0, 0);
    copies.issue(qbase, p.qs.n, q_rows, p.d, 0, 1);
    copies.issue(vbase, p.vs.n, k_rows, p.d, 0, 2);
    auto multiply = [&](auto tail_tag, f32x16 (&acc)[2][2], int t, auto&& copy) {
        const uint16_t* kt_ = lds + ring.slot(0) * WideRing::UNIT_ELEMS;
        const uint16_t* qt_ = lds + ring.slot(1) * WideRing::UNIT_ELEMS;
        if constexpr (decltype(tail_tag)::value) {
#pragma unroll
            for (int i = 0; i < 8; ++i) copy(i);
            wide_multiply_tail(acc, kt_, qt_, fk, fq, p.d - kWideStep * t);
        } else {
            wide_phase(acc, [&](int c, int u) { return *reinterpret_cast<const bf16x8*>(kt_ + (fk[u] ^ (16 * c))); },
                       [&](int c, int u) { return *reinterpret_cast<const bf16x8*>(qt_ + (fq[u] ^ (16 * c))); }, copy);
        }
        ring.next();
    };
    auto step = [&](auto tail_tag, int t) {
        const bool more = t + 1 < n_steps;
        WideRing::landed(false);                           // K and Q
        multiply(tail_tag, s, t, [&](int i) {
            if (i < 4) copies.issue(gbase, p.dos.n, q_rows, p.d, t, ring.slot(3), i);
            else if (more) copies.issue(kbase, p.ks.n, k_rows, p.d, t + 1, ring.slot(4), i - 4);
        });
        WideRing::landed(!more);                           // V and dO
        multiply(tail_tag, dp, t, [&](int i) {
            if (!more) return;
            if (i < 4) copies.issue(qbase, p.qs.n, q_rows, p.d, t + 1, ring.slot(3), i);
            else copies.issue(vbase, p.vs.n, k_rows, p.d, t + 1, ring.slot(4), i - 4);
        });
    };
    // the step that ends inside 64 behind the loop: as a choice within it, it made the compiler move both accumulators
    // (384 registers) around every step
    const int n_whole = p.d / kWideStep;
    for (int t = 0; t < n_whole; ++t) step(No{}, t);
    if (n_whole < n_steps) step(Yes{}, n_whole);
    __syncthreads();                                       // the tiles are no longer needed: P and dS take their place

    // ---- P and dS: a lane owns one query per block and four consecutive keys per register group.  Through LDS (rows of 128
    // keys, granules swizzled by the row), so that a store instruction writes whole cache lines: straight from the
    // accumulators it would touch 32 of them, 16 bytes each.
    const float c_log2 = p.scale * kLog2e;
    uint16_t* p_tile = lds;
    uint16_t* ds_tile = lds + kWideTile * kWideTile;
    static_assert(2 * kWideTile * kWideTile * 2 <= WideRing::LDS_BYTES, "P and dS of a tile fit where the ring was");
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int rq = 64 * wq + 32 * qb + n, qi = q0 + rq;
        const bool ok = qi < p.Sq;
        const float nd = rows_nd[qb], l2 = rows_l2[qb];
        const int lim = ok ? (p.causal ? min(klimit, qi + 1) : klimit) : 0;     // keys below it are attended
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int key = k0 + 64 * wk + 32 * kb + 8 * g + 4 * h;
                float pr[4], dsv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = exp2_fast(fmaf(s[kb][qb][4 * g + e], c_log2, -l2));
                    pr[e] = key + e < lim ? x : 0.f;
                    dsv[e] = key + e < lim ? x * (dp[kb][qb][4 * g + e] + nd) : 0.f;
                }
                const int at = rq * kWideTile + 8 * ((8 * wk + 4 * kb + g) ^ (rq & 15)) + 4 * h;
                *reinterpret_cast<u32x2*>(p_tile + at) = u32x2{pack_bf16(pr[0], pr[1]), pack_bf16(pr[2], pr[3])};
                *reinterpret_cast<u32x2*>(ds_tile + at) = u32x2{pack_bf16(dsv[0], dsv[1]), pack_bf16(dsv[2], dsv[3])};
            }
    }
    __syncthreads();
    const int64_t out0 = ((int64_t)slice * p.sq_pad + q0) * p.sk_pad + k0;
#pragma unroll
    for (int i = 0; i < kWideTile / 16; ++i) {
        const int row = 16 * i + (tid >> 4), g = tid & 15;
        const int at = row * kWideTile + 8 * (g ^ (row & 15));
        const int64_t to = out0 + (int64_t)row * p.sk_pad + 8 * g;
        *reinterpret_cast<u32x4*>(p.probs + to) = *reinterpret_cast<const u32x4*>(p_tile + at);
        *reinterpret_cast<u32x4*>(p.ds + to) = *reinterpret_cast<const u32x4*>(ds_tile + at);
    }
}

// ---- The three products.  Output tile: 128 columns of the head dim x 128 rows (keys of dV and dK, queries of dQ), formed
// transposed so that a lane owns one row.  Units of contraction step t: 2 t = X, 64 rows (contraction) x 128 columns of dO, Q
// or K, read transposed; 2 t + 1 = W, 64 x 128 of P or dS, read transposed (dV, dK), or 128 rows x 64 of dS, read along its
// rows (dQ).
template <bool DQ>
__device__ __forceinline__ void bwd_wide_product(const BwdWideParams& p, const uint16_t* x, const Strides& xs, const uint16_t* w, uint16_t* out,
                                                 const Strides& outs, float mul, int slice, int mt, int dt) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int wd = wave & 1, wm = wave >> 1;          // this wavefront's 64 columns of the head dim and 64 rows of the output
    const int bh = p.bh0 + slice, b = bh / p.H, hh = bh % p.H;
    const int m0 = mt * kWideTile, d0 = dt * kWideTile;
    const int n_out = DQ ? p.Sq : p.Sk, n_con = DQ ? p.Sk : p.Sq;      // rows of the output, length of the contraction
    int con_lo = 0, con_hi = DQ ? p.sk_pad : p.sq_pad;
    if (p.causal) {                                    // tiles that were not formed
        if (DQ) con_hi = min(con_hi, m0 + kWideTile);
        else con_lo = min(m0, con_hi);
    }
    const uint16_t* xbase = x + b * xs.b + hh * xs.h + d0;
    const uint16_t* wbase = w + (int64_t)slice * p.sq_pad * p.sk_pad + (DQ ? (int64_t)m0 * p.sk_pad : m0);

    // ---- copies: X: 16 of 4 rows x 256 bytes; W the same, or (DQ) 16 of 8 rows x 128 bytes
    uint32_t xoff[4], woff[4];
    int xrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = (4 * wave + i) * 4 + (lane >> 4), g = (lane & 15) ^ swz<128>(row);
        xrow[i] = row;
        xoff[i] = 2u * (uint32_t)(d0 + 8 * g < p.d ? 8 * g : 0);        // columns past the head dim: filler, not stored
        if (DQ) {
            const int wr = (4 * wave + i) * 8 + (lane >> 3), wg = (lane & 7) ^ swz<64>(wr);
            woff[i] = 2u * (uint32_t)(wr * p.sk_pad + 8 * wg);
        } else {
            woff[i] = 2u * (uint32_t)(row * p.sk_pad + 8 * g);
        }
    }
    const uint32_t lds0 = lds_addr(lds) + 4096u * (uint32_t)wave;
    auto issue_x = [&](int c0, int slot, int i) {      // copy i of contraction rows [c0, c0 + 64); past the end the last row, against zeros of W
        const int first = min(c0, n_con - 1), over = n_con - 1 - first;
        dma16u(xbase + (int64_t)first * xs.n, xoff[i] + 2u * (uint32_t)(min(xrow[i], over) * (int)xs.n), lds0 + 2u * (uint32_t)(slot * WideRing::UNIT_ELEMS) + 1024u * i);
    };
    auto issue_w = [&](int c0, int slot, int i) {
        dma16u(wbase + (DQ ? (int64_t)c0 : (int64_t)c0 * p.sk_pad), woff[i], lds0 + 2u * (uint32_t)(slot * WideRing::UNIT_ELEMS) + 1024u * i);
    };
    // fragment addresses: transposing reads of a 64 x 128 tile, 16 contraction rows per chunk
    const int tr_r = lane & 15, tr_g16 = (lane >> 4) & 1;
    // (DQ: eight consecutive contraction rows per half wave, as the row reads of dS have them; else 4 h and 8 further on)
    int xo[2][2], wo[2][2];                            // [half of the chunk][block of 32]; DQ: wo[0][block], the chunk flips bits 4 and 5
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int row = DQ ? 8 * h + (tr_r >> 2) + 4 * half : 4 * h + (tr_r >> 2) + 8 * half;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            xo[half][u] = row * 128 + 8 * ((4 * (2 * wd + u) + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<128>(row)) + 4 * (tr_r & 1);
            if (DQ) {
                const int wr = 64 * wm + 32 * u + n;
                wo[half][u] = wr * kWideStep + 8 * (h ^ swz<64>(wr));
            } else {
                wo[half][u] = row * 128 + 8 * ((4 * (2 * wm + u) + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<128>(row)) + 4 * (tr_r & 1);
            }
        }
    }
    auto tr_frag = [&](const uint16_t* tile, int o0, int o1) {
        const u32x2 lo = lds_read_tr16(tile + o0), hi = lds_read_tr16(tile + o1);
        return __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    };

    f32x16 acc[2][2];                                  // [head-dim block][row block]
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][m][r] = 0.f;

    WideRing ring;
    if (con_lo < con_hi) {
#pragma unroll
        for (int i = 0; i < 4; ++i) issue_x(con_lo, 0, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) issue_w(con_lo, 1, i);
        if (con_lo + kWideStep < con_hi)
#pragma unroll
            for (int i = 0; i < 4; ++i) issue_x(con_lo + kWideStep, 2, i);
    }
    for (int c0 = con_lo; c0 < con_hi; c0 += kWideStep, ring.next()) {
        WideRing::landed(c0 + kWideStep >= con_hi);
        const uint16_t* xt = lds + ring.slot(0) * WideRing::UNIT_ELEMS;
        const uint16_t* wt = lds + ring.slot(1) * WideRing::UNIT_ELEMS;
        wide_phase(acc, [&](int c, int u) { return tr_frag(xt + 16 * c * 128, xo[0][u], xo[1][u]); },
                   [&](int c, int u) {
                       if constexpr (DQ) return *reinterpret_cast<const bf16x8*>(wt + (wo[0][u] ^ (16 * c)));
                       else return tr_frag(wt + 16 * c * 128, wo[0][u], wo[1][u]);
                   },
                   [&](int i) {
                       if (i < 4 && c0 + kWideStep < con_hi) issue_w(c0 + kWideStep, ring.slot(3), i);
                       if (i >= 4 && c0 + 2 * kWideStep < con_hi) issue_x(c0 + 2 * kWideStep, ring.slot(4), i - 4);
                   });
    }
    __syncthreads();                                   // the tiles are no longer needed: the output passes through their place
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int row0 = m0 + 64 * wm + 32 * m, col0 = d0 + 64 * wd;
        store_rows32<64>(lds + wave * 32 * 64, out + b * outs.b + hh * outs.h + (int64_t)row0 * outs.n + col0, outs.n, n_out - row0, p.d - col0, [&](int u, int g) {
            const f32x16& a = acc[u][m];
            return u32x2{pack_bf16(a[4 * g] * mul, a[4 * g + 1] * mul), pack_bf16(a[4 * g + 2] * mul, a[4 * g + 3] * mul)};
        });
    }
}

static __global__ __launch_bounds__(256, 2) void bwd_wide_products_kernel(const BwdWideParams p) {
    const int n_kt = p.sk_pad / kWideTile, n_qt = p.sq_pad / kWideTile, n_dt = (p.d + kWideTile - 1) / kWideTile;
    const int per_slice = (2 * n_kt + n_qt) * n_dt;
    const int wg = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = wg / per_slice, j = wg % per_slice, dt = j % n_dt, m = j / n_dt;
    if (m < n_kt) bwd_wide_product<false>(p, p.dout, p.dos, p.probs, p.dv, p.dvs, 1.0f, slice, m, dt);
    else if (m < 2 * n_kt) bwd_wide_product<false>(p, p.q, p.qs, p.ds, p.dk, p.dks, p.scale, slice, m - n_kt, dt);
    else bwd_wide_product<true>(p, p.k, p.ks, p.ds, p.dq, p.dqs, p.scale, slice, m - 2 * n_kt, dt);
}

}  // namespace fattn
