// Forward for head dims above 256 where the caller has room for the probabilities of a (batch, head) slice.  O of 32 queries at
// D = 512 alone takes 256 registers per lane: the one-pass kernel (attn_fwd_bigd.hpp) has two wavefronts form the same S for
// half of O each and one MFMA per fragment that it reads from LDS.  Here the two products are matrix products of 128 x 128
// tiles, four MFMAs per four fragments, as in the backward (attn_bwd_wide.hpp, whose tiles, copies and ring these are):
//   fwd_probs_kernel    S^T = K Q^T, 128 keys x 128 queries per workgroup; P = exp2(S c - m) with the maximum m of a query over
//                       the tile's keys, stored as bf16, and m and the sum of P (fp32, before the rounding) per query and tile
//   fwd_probs_pv_kernel O^T = sum over the key tiles t of w_t V_t^T P_t, 128 columns of the head dim x 128 queries per
//                       workgroup: the online softmax over tiles, each tile's product in accumulators of its own that are
//                       scaled into the sum, so that a P is rounded relative to its own tile's maximum, and the sums are fp32
// P is [Sq, Sk] padded to multiples of 128 (zero there); the launcher takes as many slices at a time as the workspace holds.
// Tiles that the causal flag excludes are neither formed nor read.
#pragma once
#include "attn_bwd_wide.hpp"

namespace fattn {

struct FwdProbsParams {
    const uint16_t *q, *k, *v;
    uint16_t* o;
    float* lse;                   // [B*H, Sq] or null
    uint16_t* probs;              // [slices, sq_pad, sk_pad]
    float *tile_max, *tile_sum;   // [slices, n_kt, sq_pad]: maximum of S c (log2 units) and sum of P
    Strides qs, ks, vs, os;
    int B, H, Sq, Sk, d;
    int sq_pad, sk_pad;           // multiples of 128
    int bh0;                      // first (batch, head) slice of this launch
    float scale;
    const int32_t* kv_len;
    int causal;
    int key_splits = 1;           // 1: O and LSE are written directly
    float* part_o = nullptr;      // [key_splits][B*H*Sq][d]
    float* part_lse = nullptr;    // [key_splits][B*H*Sq], as in FwdParams
};

static __global__ __launch_bounds__(256, 2) void fwd_probs_kernel(const FwdProbsParams p) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int wk = wave & 1, wq = wave >> 1;          // this wavefront's 64 keys and 64 queries of the tile

    // bands of eight key tiles, query tiles across, as in bwd_wide_scores_kernel
    const int n_kt = p.sk_pad / kWideTile, n_qt = p.sq_pad / kWideTile;
    const int wg = xcd_remap_tiles(blockIdx.x, gridDim.x, n_kt * n_qt, p.causal);
    const int slice = wg / (n_kt * n_qt), in_slice = wg % (n_kt * n_qt);
    const int band = in_slice / (8 * n_qt), in_band = in_slice % (8 * n_qt), width = min(8, n_kt - 8 * band);
    const int kt = 8 * band + in_band % width, qt = in_band / width;
    const int bh = p.bh0 + slice, b = bh / p.H, hh = bh % p.H;
    const int k0 = kt * kWideTile, q0 = qt * kWideTile;
    int klimit = p.Sk;
    if (p.kv_len) klimit = min(klimit, max(p.kv_len[b], 0));
    if (k0 >= klimit || (p.causal && k0 > q0 + kWideTile - 1)) return;      // nothing of this tile is attended, and nothing reads it

    const int k_rows = p.Sk - k0, q_rows = p.Sq - q0;
    const uint16_t* kbase = p.k + b * p.ks.b + hh * p.ks.h + (int64_t)min(k0, p.Sk - 1) * p.ks.n;
    const uint16_t* qbase = p.q + b * p.qs.b + hh * p.qs.h + (int64_t)min(q0, p.Sq - 1) * p.qs.n;
    const WideRows copies(lds);
    int fk[2], fq[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int rk = 64 * wk + 32 * u + n, rq = 64 * wq + 32 * u + n;
        fk[u] = rk * kWideStep + 8 * (h ^ swz<64>(rk));
        fq[u] = rq * kWideStep + 8 * (h ^ swz<64>(rq));
    }
    f32x16 s[2][2];                                        // [key block][query block]
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][qb][r] = 0.f;

    // units of contraction step t: 2 t = K, 2 t + 1 = Q (rows of 64 elements)
    const int n_steps = (p.d + kWideStep - 1) / kWideStep, n_whole = p.d / kWideStep;
    WideRing ring;
    copies.issue(kbase, p.ks.n, k_rows, p.d, 0, 0);
    copies.issue(qbase, p.qs.n, q_rows, p.d, 0, 1);
    if (n_steps > 1) copies.issue(kbase, p.ks.n, k_rows, p.d, 1, 2);
    auto step = [&](auto tail_tag, int t) {
        WideRing::landed(t + 1 >= n_steps);
        const uint16_t* kt_ = lds + ring.slot(0) * WideRing::UNIT_ELEMS;
        const uint16_t* qt_ = lds + ring.slot(1) * WideRing::UNIT_ELEMS;
        if constexpr (decltype(tail_tag)::value) {         // the last one: nothing more to copy
            wide_multiply_tail(s, kt_, qt_, fk, fq, p.d - kWideStep * t);
        } else {
            wide_phase(s, [&](int c, int u) { return *reinterpret_cast<const bf16x8*>(kt_ + (fk[u] ^ (16 * c))); },
                       [&](int c, int u) { return *reinterpret_cast<const bf16x8*>(qt_ + (fq[u] ^ (16 * c))); },
                       [&](int i) {
                           if (i < 4 && t + 1 < n_steps) copies.issue(qbase, p.qs.n, q_rows, p.d, t + 1, ring.slot(3), i);
                           if (i >= 4 && t + 2 < n_steps) copies.issue(kbase, p.ks.n, k_rows, p.d, t + 2, ring.slot(4), i - 4);
                       });
        }
        ring.next();
    };
    for (int t = 0; t < n_whole; ++t) step(std::integral_constant<bool, false>{}, t);
    if (n_whole < n_steps) step(std::integral_constant<bool, true>{}, n_whole);
    __syncthreads();                                       // the tiles are no longer needed: P takes their place

    // ---- maximum and sum of every query over the tile's keys: a lane and its other half hold 64 of them, the neighbouring
    // wavefront (wk) the other 64
    const float c_log2 = p.scale * kLog2e;
    uint16_t* p_tile = lds;
    float* ml = reinterpret_cast<float*>(lds + kWideTile * kWideTile);       // [wk][maximum, sum][query]
    static_assert(kWideTile * kWideTile * 2 + 4 * kWideTile * 4 <= WideRing::LDS_BYTES, "P of a tile, maxima and sums fit where the ring was");
    float mx[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int rq = 64 * wq + 32 * qb + n, qi = q0 + rq;
        const int lim = (qi < p.Sq ? (p.causal ? min(klimit, qi + 1) : klimit) : 0) - k0 - 64 * wk - 4 * h;      // of this lane's keys: those below it
        float m = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[kb][qb][r] = 32 * kb + 8 * (r >> 2) + (r & 3) < lim ? s[kb][qb][r] : -INFINITY;
                m = fmaxf(m, s[kb][qb][r]);
            }
        mx[qb] = fmaxf(m, xhalf(m));
        if (h == 0) ml[(2 * wk) * kWideTile + rq] = mx[qb];
    }
    __syncthreads();
    float sum[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int rq = 64 * wq + 32 * qb + n;
        const float m = fmaxf(mx[qb], ml[(2 * (wk ^ 1)) * kWideTile + rq]);
        mx[qb] = m * c_log2;
        const float m_use = m == -INFINITY ? 0.f : mx[qb];
        float l0 = 0.f, l1 = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float pr[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) pr[e] = exp2_fast(fmaf(s[kb][qb][4 * g + e], c_log2, -m_use));
                l0 += pr[0] + pr[2];
                l1 += pr[1] + pr[3];
                const int at = rq * kWideTile + 8 * ((8 * wk + 4 * kb + g) ^ (rq & 15)) + 4 * h;
                *reinterpret_cast<u32x2*>(p_tile + at) = u32x2{pack_bf16(pr[0], pr[1]), pack_bf16(pr[2], pr[3])};
            }
        sum[qb] = l0 + l1;
        sum[qb] += xhalf(sum[qb]);
        if (wk == 1 && h == 0) ml[kWideTile + rq] = sum[qb];
    }
    __syncthreads();
    if (wk == 0 && h == 0) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            const int rq = 64 * wq + 32 * qb + n;
            const int64_t at = ((int64_t)slice * n_kt + kt) * p.sq_pad + q0 + rq;
            p.tile_max[at] = mx[qb];
            p.tile_sum[at] = sum[qb] + ml[kWideTile + rq];
        }
    }
    const int64_t out0 = ((int64_t)slice * p.sq_pad + q0) * p.sk_pad + k0;
#pragma unroll
    for (int i = 0; i < kWideTile / 16; ++i) {
        const int row = 16 * i + (tid >> 4), g = tid & 15;
        *reinterpret_cast<u32x4*>(p.probs + out0 + (int64_t)row * p.sk_pad + 8 * g) =
            *reinterpret_cast<const u32x4*>(p_tile + row * kWideTile + 8 * (g ^ (row & 15)));
    }
}

// Units of contraction step t (64 keys): 2 t = V, 64 keys x 128 columns, read transposed; 2 t + 1 = 128 queries x 64 keys of P,
// read along its rows (as dQ in bwd_wide_products_kernel).  key_splits workgroups share an output tile, each takes a range of
// the key tiles and leaves a normalised fp32 partial output with its log-sum-exp for fwd_merge_kernel: one head of a few
// thousand positions is about a hundred output tiles, and two workgroups per compute unit cover each other's waits.
static __global__ __launch_bounds__(256, 2) void fwd_probs_pv_kernel(const FwdProbsParams p) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int wd = wave & 1, wm = wave >> 1;          // this wavefront's 64 columns of the head dim and 64 queries
    const int n_kt = p.sk_pad / kWideTile, n_qt = p.sq_pad / kWideTile, n_dt = (p.d + kWideTile - 1) / kWideTile;
    // the column tiles of a query tile, which read the same P, side by side; then the query tiles, which read the same V
    const int wg = xcd_remap_split(blockIdx.x, gridDim.x);
    const int per = n_qt * n_dt, part_id = wg / per, split = part_id % p.key_splits, slice = part_id / p.key_splits;
    const int j = wg % per, dt = j % n_dt;
    const int mt = p.causal ? n_qt - 1 - j / n_dt : j / n_dt;              // causal: the longest walks first
    const int bh = p.bh0 + slice, b = bh / p.H, hh = bh % p.H;
    const int m0 = mt * kWideTile, d0 = dt * kWideTile;
    int klimit = p.Sk;
    if (p.kv_len) klimit = min(klimit, max(p.kv_len[b], 0));
    int all = (klimit + kWideTile - 1) / kWideTile;   // key tiles that were formed for these queries
    if (p.causal) all = min(all, mt + 1);
    const int share = (all + p.key_splits - 1) / p.key_splits, t_lo = min(split * share, all), t_hi = min(t_lo + share, all);
    const int con_lo = t_lo * kWideTile, con_hi = t_hi * kWideTile;

    const uint16_t* xbase = p.v + b * p.vs.b + hh * p.vs.h + d0;
    const uint16_t* wbase = p.probs + ((int64_t)slice * p.sq_pad + m0) * p.sk_pad;
    uint32_t xoff[4], woff[4];
    int xrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = (4 * wave + i) * 4 + (lane >> 4), g = (lane & 15) ^ swz<128>(row);
        xrow[i] = row;
        xoff[i] = 2u * (uint32_t)(d0 + 8 * g < p.d ? 8 * g : 0);           // columns past the head dim: filler, not stored
        const int wr = (4 * wave + i) * 8 + (lane >> 3);
        woff[i] = 2u * (uint32_t)(wr * p.sk_pad + 8 * ((lane & 7) ^ swz<64>(wr)));
    }
    const uint32_t lds0 = lds_addr(lds) + 4096u * (uint32_t)wave;
    auto issue_x = [&](int c0, int slot, int i) {      // copy i of keys [c0, c0 + 64); past the last attended one that one, against zeros of P
        const int r0 = min(c0, klimit - 1), over = klimit - 1 - r0;
        dma16u(xbase + (int64_t)r0 * p.vs.n, xoff[i] + 2u * (uint32_t)(min(xrow[i], over) * (int)p.vs.n), lds0 + 2u * (uint32_t)(slot * WideRing::UNIT_ELEMS) + 1024u * i);
    };
    auto issue_w = [&](int c0, int slot, int i) { dma16u(wbase + c0, woff[i], lds0 + 2u * (uint32_t)(slot * WideRing::UNIT_ELEMS) + 1024u * i); };
    const int tr_r = lane & 15, tr_g16 = (lane >> 4) & 1;
    int xo[2][2], wo[2];                               // [half of the chunk][block of 32 columns]; rows of P, the chunk flips bits 4 and 5
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int row = 8 * h + (tr_r >> 2) + 4 * half;
            xo[half][u] = row * 128 + 8 * ((4 * (2 * wd + u) + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<128>(row)) + 4 * (tr_r & 1);
        }
        const int wr = 64 * wm + 32 * u + n;
        wo[u] = wr * kWideStep + 8 * (h ^ swz<64>(wr));
    }

    f32x16 acc[2][2], part[2][2];                      // [head-dim block][query block]: the sum, the tile at hand
    float m_run[2], l_run[2];                          // of this lane's query in either block (log2 units)
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        m_run[m] = -INFINITY;
        l_run[m] = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][m][r] = 0.f;
    }
    // Maxima and sums of the next tile.  The wait for them, which the compiler makes one for everything in flight, is put
    // where the copies are waited for anyway.
    const float* maxima = p.tile_max + (int64_t)slice * n_kt * p.sq_pad + m0 + 64 * wm + n;
    const float* sums = p.tile_sum + (int64_t)slice * n_kt * p.sq_pad + m0 + 64 * wm + n;
    float m_next[2] = {0.f, 0.f}, l_next[2] = {0.f, 0.f};
    auto stats = [&](int t) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            m_next[m] = maxima[(int64_t)t * p.sq_pad + 32 * m];
            l_next[m] = sums[(int64_t)t * p.sq_pad + 32 * m];
        }
    };
    auto stats_landed = [&]() {
#pragma unroll
        for (int m = 0; m < 2; ++m) asm volatile("" : "+v"(m_next[m]), "+v"(l_next[m]));
    };
    WideRing ring;
    if (con_lo < con_hi) {
        stats(t_lo);
        stats_landed();
#pragma unroll
        for (int i = 0; i < 4; ++i) issue_x(con_lo, 0, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) issue_w(con_lo, 1, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) issue_x(con_lo + kWideStep, 2, i);     // a tile is two steps
    }
    auto step = [&](int c0, bool fetch_stats) {
        const bool last = c0 + kWideStep >= con_hi;
        WideRing::landed(last);
        if (fetch_stats) stats(c0 / kWideTile + 1);
        const uint16_t* xt = lds + ring.slot(0) * WideRing::UNIT_ELEMS;
        const uint16_t* wt = lds + ring.slot(1) * WideRing::UNIT_ELEMS;
        wide_phase(part,
                   [&](int c, int u) {
                       const u32x2 lo = lds_read_tr16(xt + 16 * c * 128 + xo[0][u]), hi = lds_read_tr16(xt + 16 * c * 128 + xo[1][u]);
                       return __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
                   },
                   [&](int c, int u) { return *reinterpret_cast<const bf16x8*>(wt + (wo[u] ^ (16 * c))); },
                   [&](int i) {
                       if (i < 4 && !last) issue_w(c0 + kWideStep, ring.slot(3), i);
                       if (i >= 4 && c0 + 2 * kWideStep < con_hi) issue_x(c0 + 2 * kWideStep, ring.slot(4), i - 4);
                   });
        ring.next();
    };
    for (int t = t_lo; t < t_hi; ++t) {
        float w_old[2], w_new[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const float m_new = fmaxf(m_run[m], m_next[m]), m_to = m_new == -INFINITY ? 0.f : m_new;
            w_old[m] = exp2_fast(m_run[m] - m_to);
            w_new[m] = exp2_fast(m_next[m] - m_to);
            l_run[m] = l_run[m] * w_old[m] + l_next[m] * w_new[m];
            m_run[m] = m_new;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) part[u][m][r] = 0.f;
        }
        step(t * kWideTile, t + 1 < t_hi);
        stats_landed();
        step(t * kWideTile + kWideStep, false);
        if (__any(w_old[0] != 1.f || w_old[1] != 1.f)) {
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[u][m][r] *= w_old[m];
        }
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[u][m][r] = fmaf(part[u][m][r], w_new[m], acc[u][m][r]);
    }

    // ---- O and LSE, or this range's part of them
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int row0 = m0 + 64 * wm + 32 * m, col0 = d0 + 64 * wd;
        const float l = l_run[m], inv = l > 0.f ? 1.0f / l : 0.f, lse = l > 0.f ? (m_run[m] + log2_fast(l)) * kLn2 : -INFINITY;
        const bool tells = dt == 0 && wd == 0 && h == 0 && row0 + n < p.Sq;
        if (p.key_splits > 1) {
            const int64_t prow = ((int64_t)split * p.B * p.H + bh) * p.Sq + row0;
            store_rows32_f32<64>(reinterpret_cast<float*>(lds) + wave * 32 * 64, p.part_o + prow * p.d + col0, p.d, p.Sq - row0, p.d - col0, [&](int u, int g) {
                const f32x16& a = acc[u][m];
                return f32x4{a[4 * g] * inv, a[4 * g + 1] * inv, a[4 * g + 2] * inv, a[4 * g + 3] * inv};
            });
            if (tells) p.part_lse[prow + n] = l != l ? l : lse;            // a NaN is not an empty range
        } else {
            store_rows32<64>(lds + wave * 32 * 64, p.o + b * p.os.b + hh * p.os.h + (int64_t)row0 * p.os.n + col0, p.os.n, p.Sq - row0, p.d - col0, [&](int u, int g) {
                const f32x16& a = acc[u][m];
                return u32x2{pack_bf16(a[4 * g] * inv, a[4 * g + 1] * inv), pack_bf16(a[4 * g + 2] * inv, a[4 * g + 3] * inv)};
            });
            if (p.lse && tells) p.lse[(int64_t)bh * p.Sq + row0 + n] = lse;
        }
    }
}

}  // namespace fattn
