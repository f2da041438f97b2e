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
// Tiles are copied global -> LDS by LDS-DMA in steps of 32 along the contraction, two stages, one barrier per step, and at
// least two workgroups per compute unit, so that one's wait is covered by the other.  Bound by LDS traffic: a wavefront's
// 64 x 64 tile reads 8 KiB per 8 MFMAs.
// B=1 H=1 S=4096 D=512: library GEMMs and separate passes 246 us, this 159 us; B=3 H=2 S=640 D=512, where the
// library's 15 calls kept the host busy, forward and backward: 615 -> 80 us.
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

constexpr int kWideTile = 128, kWideStep = 32;

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

// Rows of 32 elements (64 bytes, four granules): 16 consecutive rows reading the same granule hit 16 distinct bank groups.
__device__ __forceinline__ constexpr int swz_row32(int row) { return (row >> 2) & 3; }

// ---- P and dS.  Stage: [K | V | Q | dO] tiles of 128 rows x 32; wavefront w copies tensor w.
struct BwdWideScoresTile {
    static constexpr int TILE_ELEMS = kWideTile * kWideStep;
    static constexpr int STAGE_ELEMS = 4 * TILE_ELEMS;
    static constexpr int LDS_BYTES = 2 * STAGE_ELEMS * 2;
};

static __global__ __launch_bounds__(256, 2) void bwd_wide_scores_kernel(const BwdWideParams p) {
    using T = BwdWideScoresTile;
    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int wk = wave & 1, wq = wave >> 1;          // this wavefront's 64 keys and 64 queries of the tile

    const int n_kt = p.sk_pad / kWideTile, n_qt = p.sq_pad / kWideTile;
    const int wg = xcd_remap(blockIdx.x, gridDim.x);
    const int kt = wg % n_kt, qt = (wg / n_kt) % n_qt, slice = wg / (n_kt * n_qt);
    const int bh = p.bh0 + slice, b = bh / p.H, hh = bh % p.H;
    const int k0 = kt * kWideTile, q0 = qt * kWideTile;
    if (p.causal && k0 > q0 + kWideTile - 1) return;       // nothing of this tile is attended, and nothing reads it
    int klimit = p.Sk;
    if (p.kv_len) klimit = min(klimit, max(p.kv_len[b], 0));

    // ---- copies: 8 of 16 rows x 64 bytes per wavefront and step; rows past the end re-read the last one
    const bool is_q = wave >= 2;
    const Strides st = wave == 0 ? p.ks : wave == 1 ? p.vs : wave == 2 ? p.qs : p.dos;
    const uint16_t* base = (wave == 0 ? p.k : wave == 1 ? p.v : wave == 2 ? p.q : p.dout) + b * st.b + hh * st.h;
    const int row0 = is_q ? q0 : k0, row_max = (is_q ? p.Sq : p.Sk) - 1;
    base += (int64_t)min(row0, row_max) * st.n;
    const int cp_row = lane >> 2, cp_gran = lane & 3;
    uint32_t off[8];
    int gran[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = 16 * i + cp_row;
        gran[i] = cp_gran ^ swz_row32(row);
        off[i] = 2u * (uint32_t)(min(row, max(row_max - row0, 0)) * (int)st.n + 8 * gran[i]);
    }
    const uint32_t lds0 = lds_addr(lds);
    auto issue = [&](int s, int stage) {                   // contraction step s: elements [32 s, 32 s + 32)
        const uint32_t dst = lds0 + 2u * (uint32_t)(stage * T::STAGE_ELEMS + wave * T::TILE_ELEMS);
        const uint16_t* src = base + kWideStep * s;
        if (kWideStep * (s + 1) <= p.d) {
#pragma unroll
            for (int i = 0; i < 8; ++i) dma16u(src, off[i], dst + 1024u * i);
        } else {                                           // granules past the head dim: filler, zeroed before use
#pragma unroll
            for (int i = 0; i < 8; ++i) dma16u(src, kWideStep * s + 8 * gran[i] < p.d ? off[i] : off[i] - 16u * gran[i], dst + 1024u * i);
        }
    };
    int foff[2][2];                                        // [chunk of 16][block of 32 rows]: elements inside a tile, for the keys
    int goff[2][2];                                        // ... for the queries
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int rk = 64 * wk + 32 * u + n, rq = 64 * wq + 32 * u + n;
            foff[c][u] = rk * kWideStep + 8 * ((2 * c + h) ^ swz_row32(rk));
            goff[c][u] = rq * kWideStep + 8 * ((2 * c + h) ^ swz_row32(rq));
        }

    f32x16 s[2][2], dp[2][2];                              // [key block][query block]
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][qb][r] = dp[kb][qb][r] = 0.f;

    const int n_steps = (p.d + kWideStep - 1) / kWideStep;
    issue(0, 0);
    wait_vm0();
    __syncthreads();
    for (int t = 0; t < n_steps; ++t) {
        const int stage = t & 1;
        if (t + 1 < n_steps) issue(t + 1, stage ^ 1);
        uint16_t* tile = lds + stage * T::STAGE_ELEMS;
        if (kWideStep * (t + 1) > p.d) {                   // the last step of a head dim that is no multiple of 32
            const u32x4 z = {0u, 0u, 0u, 0u};
            for (int idx = tid; idx < 2 * kWideTile * 4; idx += 256) {      // granules of the Q and dO tiles
                const int which = 2 + (idx >> 9), row = (idx >> 2) & 127, g = idx & 3;
                if (kWideStep * t + 8 * g >= p.d)
                    *reinterpret_cast<u32x4*>(tile + which * T::TILE_ELEMS + row * kWideStep + 8 * (g ^ swz_row32(row))) = z;
            }
            // K and V as well: a filler must not meet a zero as an infinity
            for (int idx = tid; idx < 2 * kWideTile * 4; idx += 256) {
                const int which = idx >> 9, row = (idx >> 2) & 127, g = idx & 3;
                if (kWideStep * t + 8 * g >= p.d)
                    *reinterpret_cast<u32x4*>(tile + which * T::TILE_ELEMS + row * kWideStep + 8 * (g ^ swz_row32(row))) = z;
            }
            __syncthreads();
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            bf16x8 kf[2], vf[2], qf[2], gf[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                kf[u] = *reinterpret_cast<const bf16x8*>(tile + foff[c][u]);
                vf[u] = *reinterpret_cast<const bf16x8*>(tile + T::TILE_ELEMS + foff[c][u]);
                qf[u] = *reinterpret_cast<const bf16x8*>(tile + 2 * T::TILE_ELEMS + goff[c][u]);
                gf[u] = *reinterpret_cast<const bf16x8*>(tile + 3 * T::TILE_ELEMS + goff[c][u]);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) {
                    s[kb][qb] = mfma32(kf[kb], qf[qb], s[kb][qb]);
                    dp[kb][qb] = mfma32(vf[kb], gf[qb], dp[kb][qb]);
                }
        }
        wait_vm0();
        __syncthreads();
    }

    // ---- P and dS: a lane owns one query per block and four consecutive keys per register group
    const float c_log2 = p.scale * kLog2e;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int qi = q0 + 64 * wq + 32 * qb + n;
        const bool ok = qi < p.Sq;
        const float nd = ok ? p.ndelta[(int64_t)bh * p.Sq + qi] : 0.f, l2 = ok ? p.lse2[(int64_t)bh * p.Sq + qi] : INFINITY;
        const int lim = ok ? (p.causal ? min(klimit, qi + 1) : klimit) : 0;     // keys below it are attended
        const int64_t row = ((int64_t)slice * p.sq_pad + qi) * p.sk_pad;
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
                *reinterpret_cast<u32x2*>(p.probs + row + key) = u32x2{pack_bf16(pr[0], pr[1]), pack_bf16(pr[2], pr[3])};
                *reinterpret_cast<u32x2*>(p.ds + row + key) = u32x2{pack_bf16(dsv[0], dsv[1]), pack_bf16(dsv[2], dsv[3])};
            }
    }
}

// ---- The three products.  Output tile: 128 columns of the head dim x 128 rows (keys of dV and dK, queries of dQ), formed
// transposed so that a lane owns one row.  Stage: [X | W]: X = 32 rows (contraction) x 128 columns of dO, Q or K, read
// transposed; W = 32 x 128 of P or dS, read transposed (dV, dK), or 128 rows x 32 of dS, read along its rows (dQ).
struct BwdWideProductsTile {
    static constexpr int TILE_ELEMS = kWideTile * kWideStep;
    static constexpr int STAGE_ELEMS = 2 * TILE_ELEMS;
    static constexpr int LDS_BYTES = 2 * STAGE_ELEMS * 2;
};

template <bool DQ>
__device__ __forceinline__ void bwd_wide_product(const BwdWideParams& p, const uint16_t* x, const Strides& xs, const uint16_t* w, uint16_t* out,
                                                 const Strides& outs, float mul, int slice, int mt, int dt) {
    using T = BwdWideProductsTile;
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

    // ---- copies: X: 8 of 4 rows x 256 bytes; W the same, or (DQ) 8 of 16 rows x 64 bytes; four of the sixteen per wavefront
    uint32_t xoff[2], woff[2];
    int xrow[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = (2 * wave + i) * 4 + (lane >> 4), g = (lane & 15) ^ swz<128>(row);
        xrow[i] = row;
        xoff[i] = 2u * (uint32_t)(d0 + 8 * g < p.d ? 8 * g : 0);        // columns past the head dim: filler, not stored
        if (DQ) {
            const int wr = (2 * wave + i) * 16 + (lane >> 2), wg = (lane & 3) ^ swz_row32(wr);
            woff[i] = 2u * (uint32_t)(wr * p.sk_pad + 8 * wg);
        } else {
            woff[i] = 2u * (uint32_t)(row * p.sk_pad + 8 * g);
        }
    }
    const uint32_t lds0 = lds_addr(lds);
    auto issue = [&](int c0, int stage) {              // contraction rows [c0, c0 + 32); past the end the last row, against zeros of W
        const uint32_t dst = lds0 + 2u * (uint32_t)(stage * T::STAGE_ELEMS) + 2048u * (uint32_t)wave;
        const int first = min(c0, n_con - 1);
        const uint16_t* xsrc = xbase + (int64_t)first * xs.n;
        const uint16_t* wsrc = wbase + (DQ ? (int64_t)c0 : (int64_t)c0 * p.sk_pad);
        const int over = n_con - 1 - first;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            dma16u(xsrc, xoff[i] + 2u * (uint32_t)(min(xrow[i], over) * (int)xs.n), dst + 1024u * i);
            dma16u(wsrc, woff[i], dst + 2u * T::TILE_ELEMS + 1024u * i);
        }
    };
    // fragment addresses: transposing reads of a 32 x 128 tile, 16 contraction rows per chunk
    const int tr_r = lane & 15, tr_g16 = (lane >> 4) & 1;
    // (DQ: eight consecutive contraction rows per half wave, as the row reads of dS have them; else 4 h and 8 further on)
    int xo[2][2], wo[2][2];                            // [half of the chunk][block of 32]; DQ: wo[chunk][block]
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int row = DQ ? 8 * h + (tr_r >> 2) + 4 * half : 4 * h + (tr_r >> 2) + 8 * half;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            xo[half][u] = row * 128 + 8 * ((4 * (2 * wd + u) + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<128>(row)) + 4 * (tr_r & 1);
            if (DQ) {
                const int wr = 64 * wm + 32 * u + n;
                wo[half][u] = wr * kWideStep + 8 * ((2 * half + h) ^ swz_row32(wr));
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

    if (con_lo < con_hi) {
        issue(con_lo, 0);
        wait_vm0();
        __syncthreads();
    }
    int stage = 0;
    for (int c0 = con_lo; c0 < con_hi; c0 += kWideStep, stage ^= 1) {
        if (c0 + kWideStep < con_hi) issue(c0 + kWideStep, stage ^ 1);
        const uint16_t* xt = lds + stage * T::STAGE_ELEMS;
        const uint16_t* wt = xt + T::TILE_ELEMS;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            bf16x8 xf[2], wf[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                xf[u] = tr_frag(xt + 16 * c * 128, xo[0][u], xo[1][u]);
                if constexpr (DQ) {
                    wf[u] = *reinterpret_cast<const bf16x8*>(wt + wo[c][u]);
                } else {
                    wf[u] = tr_frag(wt + 16 * c * 128, wo[0][u], wo[1][u]);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int m = 0; m < 2; ++m) acc[u][m] = mfma32(xf[u], wf[m], acc[u][m]);
        }
        wait_vm0();
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int row = m0 + 64 * wm + 32 * m + n;
        if (row >= n_out) continue;
        uint16_t* orow = out + b * outs.b + hh * outs.h + (int64_t)row * outs.n;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int col = d0 + 64 * wd + 32 * u + 8 * g + 4 * h;
                const f32x16& a = acc[u][m];
                if (col < p.d)
                    *reinterpret_cast<u32x2*>(orow + col) = u32x2{pack_bf16(a[4 * g] * mul, a[4 * g + 1] * mul), pack_bf16(a[4 * g + 2] * mul, a[4 * g + 3] * mul)};
            }
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
