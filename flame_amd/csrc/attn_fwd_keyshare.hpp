// Forward for problems with few query tiles: a few new rows of a decoder against the keys and values of all earlier ones,
// or short and few sequences in general, and the last round of a large grid.  A workgroup takes 32 queries of one (batch,
// head) and its four or eight wavefronts share the keys: each walks every fourth or eighth 32-key tile on its own (an LDS
// stage of its own, no barrier in the loop), and the partial softmaxes meet in LDS at the end.  Against fwd_kernel (128 queries
// per workgroup, every wavefront walks all keys) a problem becomes four times as many workgroups with an eighth of the
// walk, which is what a grid that does not fill the chip needs; K and V are read four times as often, from L2 mostly.
// With one query tile the kernel is bound by reading K and V once; all 32 query columns of the MFMAs are computed whatever
// Sq is, the matrix cores being far from busy then.  Where even these workgroups leave compute units idle the keys are
// split over workgroups as well (FwdParams::key_splits) and fwd_merge_kernel combines the slices.
// A wavefront has one stage: the copies of its next K tile start when this one's fragments are in registers, those of V behind
// the products, so that each is in flight for half a step, and the second wavefront of the SIMD covers the rest.  (Four
// wavefronts with two stages each, one per SIMD, waited on every dependent step of the softmax alone: 256 workgroups of 32
// queries, 1536 keys, D = 128 23.7 -> 18.2 us, 160 with 2560 keys 31.9 -> 20.4 us; D = 64, 256 with 1024 keys 11.3 -> 8.8 us.
// 64 heads, one row, 4097 keys: 5.3 TB/s either way.)  The first K tile is requested ahead of Q, whose latency it shares.
#pragma once
#include "attn_fwd.hpp"

namespace fattn {

template <int D, int NW_>
struct FwdKeyShareTile {
    static constexpr int BQ = 32, BN = 32, NW = NW_;
    static constexpr int RS = kRowPitch<D>;                            // LDS row stride, elements
    static constexpr int TILE_ELEMS = BN * RS;                         // K or V
    static constexpr int ROWS_PER_DMA = 1024 / (RS * 2);
    static constexpr int NDMA = BN / ROWS_PER_DMA;                     // copies per tile and tensor
    static constexpr int O_STRIDE = D + 4;                             // floats; row stride of the partial outputs in LDS
    static constexpr int WAVE_ELEMS = BQ * (RS + 4) * 2;               // a wavefront's K and V tile; its partial output after the walk
    static constexpr int ML_FLOATS = NW * BQ * 2;                      // per wavefront and query: maximum and sum
    static constexpr int LDS_BYTES = NW * WAVE_ELEMS * 2 + ML_FLOATS * 4;
    static_assert(2 * TILE_ELEMS <= WAVE_ELEMS && BQ * O_STRIDE * 2 <= WAVE_ELEMS && WAVE_ELEMS * 2 % 512 == 0, "both fit");
};

// DROP (DropMode) as in fwd_kernel.  At D = 64 four wavefronts per SIMD, two workgroups of eight per unit; the draw by tiles takes 184 registers
// and keeps to two: within 128 it spilled 56 bytes per lane (us, that -> this: 4 heads of 512 11.8 -> 10.1, 8 of 1024 19.5 -> 15.4, 16 of 1024 33.3 -> 26.4, 2 of 4096
// 57.7 -> 45.7, 64 heads, 20 queries, 2000 keys 36.4 -> 25.3).
template <int D, int NW_, int DROP>
__global__ __launch_bounds__(64 * NW_, D == 64 && DROP != kDropTiled ? 4 : 2) void fwd_keyshare_kernel(const FwdParams p) {
    using T = FwdKeyShareTile<D, NW_>;
    constexpr int BN = T::BN, NW = T::NW, RS = T::RS, DC = D / 16, DB = D / 32, GPR = RS / 8, NDMA = T::NDMA;

    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;

    const int n_qt = (p.Sq + T::BQ - 1) / T::BQ;
    const int all = xcd_remap(blockIdx.x, gridDim.x);            // the workgroups of a (batch, head) share an L2
    const int slice = all % p.key_splits, wg = p.wg_base + all / p.key_splits;
    const int bh = wg / n_qt, qi = (wg % n_qt) * T::BQ + n, q0 = (wg % n_qt) * T::BQ;     // qi: this lane's query
    const int b = bh / p.H, hh = bh % p.H;
    const uint16_t* qbase = p.q + b * p.qs.b + hh * p.qs.h;
    const uint16_t* kbase = p.k + b * p.ks.b + hh * p.ks.h;
    const uint16_t* vbase = p.v + b * p.vs.b + hh * p.vs.h;

    int klimit = p.Sk;
    if (p.m.kv_len) klimit = min(klimit, max(p.m.kv_len[b], 0));
    int kend = klimit;
    if (p.m.causal) kend = min(kend, q0 + T::BQ);
    const int n_tiles_all = (kend + BN - 1) / BN;
    const int per = (n_tiles_all + p.key_splits - 1) / p.key_splits;
    const int t_lo = slice * per, t_hi = min(n_tiles_all, t_lo + per);

    // ---- tile copies: this wavefront's tiles are t_lo + wave, + NW, ...
    uint16_t* const ks = lds + wave * T::WAVE_ELEMS;
    uint16_t* const vs = ks + T::TILE_ELEMS;
    const uint32_t k_dst = lds_addr(ks), v_dst = lds_addr(vs);
    const int row_in = lane / GPR, gran = lane % GPR;
    uint32_t k_lane_off[NDMA], v_lane_off[NDMA];                // bytes
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int row = i * T::ROWS_PER_DMA + row_in;
        const int c = gran ^ swz<D>(row);
        k_lane_off[i] = 2u * (uint32_t)(row * (int)p.ks.n + src_granule(c, p.d) * 8);
        v_lane_off[i] = 2u * (uint32_t)(row * (int)p.vs.n + src_granule(c, p.dv) * 8);
    }
    auto issue_rows = [&](const uint16_t* base, int64_t row_stride, const uint32_t (&lane_off)[NDMA], uint32_t dst, int t) {
        const uint16_t* tile = base + (int64_t)t * BN * row_stride;
        const int row_max = klimit - 1 - t * BN;                 // not negative for a tile that is walked
        if (row_max >= BN - 1) {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) dma16u(tile, lane_off[i], dst + 1024u * i);
        } else {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) {  // rows past the attended range re-read the last attended key, `over` rows further up
                const int over = max(i * T::ROWS_PER_DMA + row_in - row_max, 0);
                dma16u(tile, lane_off[i] - 2u * (uint32_t)(over * (int)row_stride), dst + 1024u * i);
            }
        }
    };
    auto issue_k = [&](int t) { issue_rows(kbase, p.ks.n, k_lane_off, k_dst, t); };
    auto issue_v = [&](int t) { issue_rows(vbase, p.vs.n, v_lane_off, v_dst, t); };

    // ---- the first K tile and, behind it, the Q fragments (B operand of S^T = K Q^T): column = query, 8 consecutive d.
    // Q passes through the place of the V tile.
    int t = t_lo + wave;
    if (t < t_hi) issue_k(t);
    bf16x8 qf[DC];
    {
        u32x4 w[DC];
        load_rows32<D>(w, qbase + (int64_t)q0 * p.qs.n, p.qs.n, p.Sq - q0, p.d);
        fragments_of_rows32<D>(vs, w, [&](auto dc, u32x4 f) { qf[decltype(dc)::value] = __builtin_bit_cast(bf16x8, f); });
    }
    // the fragments have been read before the first copies overwrite their place, and the compiler's wait for the loads above
    // does not become one for those copies
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) asm volatile("" : "+v"(qf[dc]));
    wait_lds_reads<0>();
    __builtin_amdgcn_sched_barrier(0);
    if (t < t_hi) issue_v(t);

    int koff[DC];
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) koff[dc] = n * RS + (((2 * dc + h) ^ swz<D>(n)) << 3);
    const int tr_r = lane & 15, tr_g16 = (lane >> 4) & 1;
    int voff[2][DB];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int row = 4 * h + (tr_r >> 2) + 8 * half;
#pragma unroll
        for (int db = 0; db < DB; ++db)
            voff[half][db] = row * RS + (((4 * db + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<D>(row)) << 3) + 4 * (tr_r & 1);
    }

    const float c_log2 = p.scale * kLog2e;
    float m_run = -INFINITY, l_run = 0.f, l_odd = 0.f;      // both halves of a wave hold the same maximum, each its own part of the sum
    f32x16 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
    const uint32_t drop_row = ((uint32_t)bh * (uint32_t)p.Sq + (uint32_t)qi) * (uint32_t)p.Sk + 4u * (uint32_t)h;

    for (; t < t_hi; t += NW) {
        const bool more = t + NW < t_hi;
        wait_vm<NDMA>();                               // K has landed, V may still be in flight
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 kf[DC];
#pragma unroll
        for (int dc = 0; dc < DC; ++dc) kf[dc] = *reinterpret_cast<const bf16x8*>(ks + koff[dc]);
#pragma unroll
        for (int dc = 0; dc < DC; ++dc) asm volatile("" : "+v"(kf[dc]));
        wait_lds_reads<0>();                           // the next copies overwrite what these reads have returned
        __builtin_amdgcn_sched_barrier(0);
        if (more) issue_k(t + NW);
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int dc = 0; dc < DC; ++dc) s = mfma32(kf[dc], qf[dc], s);
        const int lim = (p.m.causal ? min(klimit, qi + 1) : klimit) - t * BN - 4 * h;
        if (__any(lim < BN))
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) >= lim ? -INFINITY : s[r];
        float tmax = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
        if (__any(tmax > m_run)) {                     // each half tests its own keys
            tmax = max_of_halves(tmax);
            const float m_new = fmaxf(m_run, tmax);
            const float m_to = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = exp2_fast((m_run - m_to) * c_log2);
            m_run = m_new;
            l_run *= alpha;
            l_odd *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        }
        const float msc = ((m_run == -INFINITY) ? 0.f : m_run) * c_log2;
        const uint32_t drop_tile = drop_row + (uint32_t)(t * BN), drop_word = DROP == kDropRows64 ? xorshift32(p.m.drop_seed ^ drop_tile) : 0u;
        (void)drop_tile;
        (void)drop_word;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = exp2_fast(fmaf(s[r], c_log2, -msc));
            if (r & 1) l_odd += s[r];
            else l_run += s[r];
            if constexpr (DROP == kDropTiled)
                s[r] *= drop_factor_at(p.m, (uint32_t)bh, (uint32_t)qi, (uint32_t)(t * BN + acc_row(r, h)), (uint32_t)p.Sq, (uint32_t)p.Sk);
            if constexpr (DROP == kDropFlat || DROP == kDropRows64) {
                const uint32_t off = 8 * (r >> 2) + (r & 3);
                const uint32_t w = DROP == kDropRows64 ? drop_word ^ xorshift32(off) : xorshift32(p.m.drop_seed ^ (drop_tile + off));
                s[r] = w >= p.m.drop_thr32 ? s[r] : 0.f;
            }
        }
        bf16x8 pf[2];
        pf[0] = pack8(s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]);
        pf[1] = pack8(s[8], s[9], s[10], s[11], s[12], s[13], s[14], s[15]);
        if (more) wait_vm<NDMA>();                     // V has landed, the next K may still be in flight
        else wait_vm<0>();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const u32x2 lo = lds_read_tr16(vs + voff[0][db] + 16 * cc * RS);
                const u32x2 hi = lds_read_tr16(vs + voff[1][db] + 16 * cc * RS);
                const u32x4 u = {lo[0], lo[1], hi[0], hi[1]};
                oacc[db] = mfma32(__builtin_bit_cast(bf16x8, u), pf[cc], oacc[db]);
            }
        // the copies of the next tile overwrite this one: its reads have returned (their MFMAs were issued)
        __builtin_amdgcn_sched_barrier(0);
        wait_lds_reads<0>();
        if (more) issue_v(t + NW);
    }
    l_run += l_odd;

    // ---- the wavefronts' partial softmaxes meet: unnormalised O, maximum and sum of every query row
    float* ml = reinterpret_cast<float*>(lds + NW * T::WAVE_ELEMS);             // [wave][query][maximum, sum]
    {
        const float l = l_run + xhalf(l_run);
        float* orow = reinterpret_cast<float*>(ks) + n * T::O_STRIDE;
        if (qi < p.Sq && t_lo + wave < t_hi) {
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<f32x4*>(orow + 32 * db + 8 * g + 4 * h) =
                        f32x4{oacc[db][4 * g], oacc[db][4 * g + 1], oacc[db][4 * g + 2], oacc[db][4 * g + 3]};
            if (h == 0) {
                ml[(wave * T::BQ + n) * 2] = m_run;
                ml[(wave * T::BQ + n) * 2 + 1] = l;
            }
        }
    }
    __syncthreads();
    const int walked = min(NW, t_hi - t_lo);       // wavefronts with a tile
    const int groups = p.dv >> 2;                  // columns in fours
    const int64_t rows = (int64_t)p.B * p.H * p.Sq;
    for (int idx = tid; idx < min(T::BQ, p.Sq - q0) * groups; idx += 64 * NW) {
        const int row = idx / groups, g = idx % groups;
        float m = -INFINITY;
        for (int w = 0; w < walked; ++w) m = fmaxf(m, ml[(w * T::BQ + row) * 2]);
        const float m_to = (m == -INFINITY) ? 0.f : m;
        float l = 0.f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < walked; ++w) {
            const float a = exp2_fast((ml[(w * T::BQ + row) * 2] - m_to) * c_log2);
            const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(lds + w * T::WAVE_ELEMS) + row * T::O_STRIDE + 4 * g);
            l = fmaf(a, ml[(w * T::BQ + row) * 2 + 1], l);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = fmaf(a, v[i], acc[i]);
        }
        float inv = l > 0.f ? 1.0f / l : 0.f;
        if constexpr (DROP == kDropFlat || DROP == kDropRows64) inv *= p.m.drop_scale;
        const float lse = l > 0.f ? (m * c_log2 + log2_fast(l)) * kLn2 : -INFINITY;
        const int64_t r = (int64_t)bh * p.Sq + q0 + row;
        if (p.key_splits > 1) {
            *reinterpret_cast<f32x4*>(p.part_o + ((int64_t)slice * rows + r) * p.dv + 4 * g) = f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
            if (g == 0) p.part_lse[(int64_t)slice * rows + r] = l != l ? l : lse;      // a NaN is not an empty slice
        } else {
            uint16_t* orow = p.o + b * p.os.b + hh * p.os.h + (int64_t)(q0 + row) * p.os.n;
            *reinterpret_cast<u32x2*>(orow + 4 * g) = u32x2{pack_bf16(acc[0] * inv, acc[1] * inv), pack_bf16(acc[2] * inv, acc[3] * inv)};
            if (p.lse && g == 0) p.lse[r] = lse;
        }
    }
}

}  // namespace fattn
