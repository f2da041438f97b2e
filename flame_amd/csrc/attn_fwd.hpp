// Tiled QK^T -> online softmax -> PV forward for gfx950.  Writes O (bf16) and, when asked, the
// per-row log-sum-exp of the scaled logits; the Sq x Sk score matrix never leaves registers.
//
// One workgroup = NW wavefronts (4 or 8) = 32*NW query rows of one (batch, head); each wavefront owns
// 32 rows whose Q fragments stay in registers.  Eight wavefronts share each K/V tile among twice as
// many queries (half the copy traffic per MFMA) and are used when the query count fills such
// workgroups; either way two wavefronts are resident per SIMD.  K/V tiles of 64 keys are copied global -> LDS
// by the asynchronous LDS-DMA loads (no staging registers), double buffered, row-major with an XOR
// swizzle of the 16-byte granules so that both the row reads of K and the transposing reads of V are
// free of bank conflicts without padding.  The logits are produced transposed, S^T = K Q^T, so that
// every lane holds values of a single query: row max / row sum are in-lane reductions plus one
// exchange between the wave halves, the bf16 P^T values are already in the B-operand layout of the
// second MFMA (O^T = V^T P^T), and the running rescale of O is a per-lane scalar that is skipped
// while the running maximum stays within 2^8 of the reference maximum in use.
//
// The key loop is software-pipelined inside each wavefront: a wavefront issues at most one
// instruction every four cycles, and the matrix pipe and the vector ALU only run side by side when
// their instructions alternate in that stream.  Step t therefore threads the exponentials of tile t
// between the MFMAs that produce the logits of tile t+1, and the row-maximum scan of tile t+1 between
// the MFMAs of O += P(t) V(t).  The K tile in LDS runs one tile ahead of the V tile.
#pragma once
#include <type_traits>

#include "attn_common.hpp"

namespace fattn {

struct FwdParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* o;
    float* lse;          // contiguous [B*H, Sq] or null
    Strides qs, ks, vs, os;
    int B, H, Sq, Sk;
    int d;               // real head dim of Q and K: a multiple of 8, at most the compiled D
    int dv;              // real head dim of V and O, likewise
    float scale;
    MaskArgs m;
    int wg_base = 0;     // the launch covers the problem's workgroups from this one on (problems without exclusions only)
    // Key split (the key-sharing forward and the one for head dims above 128): key_splits workgroups share a query tile, each walks a contiguous slice of its key tiles and leaves a
    // normalised fp32 partial output with its log-sum-exp; fwd_merge_kernel combines them.
    int key_splits = 1;          // 1: O and LSE are written directly
    float* part_o = nullptr;     // [key_splits][B*H*Sq][dv]
    float* part_lse = nullptr;   // [key_splits][B*H*Sq], natural log, -inf for a slice without an attended key, NaN for one with a NaN
};

template <int D>
struct FwdTile {
    static constexpr int BN = 64;                   // keys per tile
    static constexpr int RS = kRowPitch<D>;         // LDS row stride, elements
    static constexpr int TILE_ELEMS = BN * RS;      // one K or V tile
    static constexpr int STAGE_ELEMS = 2 * TILE_ELEMS;
    static constexpr int LDS_BYTES = 2 * STAGE_ELEMS * 2;
    static constexpr int BIAS_PASS_BYTES = 4 * 2048;             // behind the stages: 2 KiB per wavefront that bias rows pass through
    static constexpr int ROWS_PER_DMA = 1024 / (RS * 2);         // rows covered by one 64-lane x 16-byte copy
    static constexpr int DMA_PER_WAVE = BN / ROWS_PER_DMA / 4;   // copies per wave and tensor
    // Q passes through the place of a V tile, 2 KiB per wavefront; behind the stages where a tile is smaller than that
    static constexpr int q_pass_bytes(int nw) { return nw * 2048 > TILE_ELEMS * 2 ? nw * 2048 : 0; }
};

// 16 bytes of a bias row, at any element's address
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x8_any __attribute__((ext_vector_type(8), aligned(2)));

// DROP (DropMode): the probabilities that multiply V are dropped element by element (drop_factor) and O is rescaled; the
// row sums, and with them the log-sum-exp, stay those of the undropped softmax.
// KG = 2: two groups of NW wavefronts share the workgroup's queries, each walks one half of the key tiles in LDS stages of its
// own, and the second hands its running state to the first through LDS.  For grids that give a compute unit one workgroup at
// most: its second wavefront per SIMD, which otherwise a second workgroup would be, and half the walk.  K and V are still
// read once per workgroup.
// AHEAD: a bias is requested a step earlier (see EARLY).
// DEALT: the units come in the order of causal_order.hpp (deals_units, which the host asks).
template <int D, int EXCL, int NW, int DROP, int KG, bool AHEAD, bool DEALT>
__device__ __forceinline__ void fwd_body(const FwdParams& p) {
    static_assert(KG == 1 || (KG == 2 && EXCL == kExNone), "key groups: nothing excluded but by causal flag and key lengths");
    static_assert(!DEALT || (KG == 1 && DROP == kDropNone), "more than one workgroup per compute unit, no dropout");
    using T = FwdTile<D>;
    constexpr int BN = T::BN, RS = T::RS;
    constexpr int BM = 32 * NW;  // query rows per workgroup
    constexpr int DC = D / 16;   // contraction chunks of QK^T
    constexpr int DB = D / 32;   // 32-row blocks of O^T
    constexpr int GPR = RS / 8;  // 16-byte granules per row in LDS
    constexpr int NDMA = T::DMA_PER_WAVE * 4 / NW;
    constexpr int PD = 4;        // LDS read-ahead depth, in fragments
    // Tile t lives in stage t % 2; K runs 2 tiles and V 1 tile ahead of use, one barrier per step.
    // (Measured: four stages with counted waits, or a barrier only every second step, are not faster, not even for a
    // workgroup that has its compute unit to itself: the step is bound by instruction issue, not by the copies.)
    constexpr int KD = 2, VD = 1;
    static_assert((2 * DC) % PD == 0 && (4 * DB) % PD == 0, "read-ahead depth must divide the fragment counts");

    extern __shared__ __attribute__((aligned(1024))) uint16_t lds_all[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = KG == 1 ? wave_all : wave_all % NW, group = KG == 1 ? 0 : wave_all / NW;
    const int n = lane & 31, h = lane >> 5;
    uint16_t* lds = lds_all + (KG == 1 ? 0 : group * (T::LDS_BYTES / 2));

    const int n_qt = (p.Sq + BM - 1) / BM;
    constexpr bool KNOWS_BIAS = EXCL == kExBiasF32 || EXCL == kExBiasBf16;       // no causal flag, no key lengths
    const bool falling = !KNOWS_BIAS && EXCL != kExKeys && p.m.causal && !p.m.kv_len;
    const bool by_batch = !KNOWS_BIAS && (p.m.kv_len || EXCL == kExKeys || EXCL == kExBits);
    const int wg = p.wg_base + xcd_remap_heads<NW == 4 && KG == 1 && EXCL != kExBits>(blockIdx.x, gridDim.x, n_qt, by_batch, falling);
    int qt = wg % n_qt, bh = wg / n_qt;
    if constexpr (DEALT) {
        int t, s;
        dealt_unit<NW == 4 && EXCL != kExBits>(blockIdx.x, n_qt, p.B, p.H, !falling, t, s);
        qt = __builtin_amdgcn_readfirstlane(falling ? n_qt - 1 - t : t);         // (the compiler divides in vector registers)
        bh = __builtin_amdgcn_readfirstlane(s);
    } else if (falling) {
        causal_longest_first<NW == 4 && KG == 1>(wg, n_qt, gridDim.x, qt, bh);
    }
    if (EXCL == kExKeys || (p.m.kv_len && EXCL != kExBits)) bh = longest_batches_first<EXCL == kExKeys>(bh, p.B, p.H, p.Sk, p.m);
    // a bias that all batches share: its rows are read by the batches' workgroups one after the other on one XCD, from its L2
    if ((EXCL == kExBiasF32 || EXCL == kExBiasBf16) && p.m.bb == 0) {
        const int rest = wg / p.B;
        qt = rest % n_qt;
        bh = (wg % p.B) * p.H + rest / n_qt;
    }
    const int b = bh / p.H, hh = bh % p.H;
    const int q0 = qt * BM;
    const int qw0 = q0 + wave * 32;
    const int qi = qw0 + n;                           // this lane's query

    const uint16_t* qbase = p.q + b * p.qs.b + hh * p.qs.h;
    const uint16_t* kbase = p.k + b * p.ks.b + hh * p.ks.h;
    const uint16_t* vbase = p.v + b * p.vs.b + hh * p.vs.h;

    int klimit = p.Sk;
    if (p.m.kv_len) klimit = min(klimit, max(p.m.kv_len[b], 0));
    int kend = klimit;
    if (p.m.causal) kend = min(kend, q0 + BM);
    int n_tiles = (kend + BN - 1) / BN;
    // The tiles of this wavefront's group become tiles 0 .. n_tiles - 1 of a walk that starts at key `key0`.
    const int n_first = (n_tiles + 1) / 2;            // of group 0
    const int key0 = KG == 1 ? 0 : group * n_first * BN;
    if constexpr (KG == 2) {
        n_tiles = group ? n_tiles - n_first : n_first;
        klimit -= key0;
        kbase += key0 * p.ks.n;
        vbase += key0 * p.vs.n;
    }
    const uint8_t* mbase = (EXCL != kExNone && p.m.mask) ? mask_head_base(p.m, b, hh) : nullptr;
    const char* bbase = (EXCL == kExGeneral && p.m.bias)
                            ? static_cast<const char*>(p.m.bias) + (b * p.m.bb + hh * p.m.bh) * (p.m.bias_f32 ? 4 : 2)
                            : nullptr;

    // KEYS: step t of the walk takes tile tile_of(t) (elsewhere the two are the same number); stages go by the step
    constexpr bool BITS = EXCL == kExBits, KEYS = EXCL == kExKeys || BITS;
    KeyTiles kt;
    const uint64_t* brows = nullptr;               // BITS: words of key tile 0, one per query; tiles lie 64 bit_nqt words apart
    if constexpr (BITS) {
        const int plane = b * p.m.plane_b + hh * p.m.plane_h;
        const uint8_t* flags = p.m.tile_flags + ((int64_t)plane * p.m.bit_nqt + q0 / 64) * p.m.bit_nkt;       // of the first 64 queries, then of the others
        kt.build_of_tiles(reinterpret_cast<char*>(lds) + T::LDS_BYTES, (klimit + 63) / 64, [&](int t) {
            const int f0 = flags[t], f1 = flags[p.m.bit_nkt + t];
            return f0 & f1 & kTileAllKeys ? 2 : (f0 | f1) & kTileAny ? 1 : 0;
        });
        n_tiles = kt.n_tiles;
        brows = p.m.bit_rows + (int64_t)plane * p.m.bit_nkt * (64 * p.m.bit_nqt);
    } else if constexpr (KEYS) {
        kt.build(reinterpret_cast<char*>(lds) + T::LDS_BYTES, klimit, NW, [&](int key) {
            return key < klimit && mask_attends(p.m, mbase, (int64_t)min(key, p.Sk - 1) * p.m.sk);
        });
        n_tiles = kt.n_tiles;
    }
    auto tile_of = [&](int t) {
        if constexpr (KEYS) return kt.tile(t);
        else return t;
    };
    constexpr bool BIAS = EXCL == kExBiasF32 || EXCL == kExBiasBf16;

    // ---- asynchronous tile copies.  Full tiles: uniform tile base + a per-lane 32-bit byte offset that never changes;
    //      ragged tiles clamp their rows into the attended range.
    const uint32_t lds0 = lds_addr(lds);
    const int dma_row_in = lane / GPR;                       // row inside one 1 KiB copy
    const int dma_gran = lane % GPR;                         // physical granule written by this lane
    uint32_t k_lane_off[NDMA], v_lane_off[NDMA];
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int row = (wave * NDMA + i) * T::ROWS_PER_DMA + dma_row_in;
        const int c = dma_gran ^ swz<D>(row);
        k_lane_off[i] = 2u * (uint32_t)(row * (int)p.ks.n + src_granule(c, p.d) * 8);
        v_lane_off[i] = 2u * (uint32_t)(row * (int)p.vs.n + src_granule(c, p.dv) * 8);
    }
    auto dst_of = [&](int t, int which, int i) {             // LDS byte address of copy i of this wave
        return lds0 + 2u * (uint32_t)((t & 1) * T::STAGE_ELEMS + which * T::TILE_ELEMS + (wave * NDMA + i) * 512);
    };
    // any tile: rows past the attended range re-read the last attended key, which lies `over` rows further up
    const int dma_row0 = wave * NDMA * T::ROWS_PER_DMA + dma_row_in;
    auto issue_any = [&](const uint16_t* base, int64_t row_stride, const uint32_t (&lane_off)[NDMA], int t, int which) {
        const int tile = tile_of(t);
        const uint16_t* tb = base + (int64_t)tile * BN * row_stride;
        const int row_max = klimit - 1 - tile * BN;          // not negative for a tile that is walked
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int over = max(dma_row0 + i * T::ROWS_PER_DMA - row_max, 0);
            dma16u(tb, lane_off[i] - 2u * (uint32_t)(over * (int)row_stride), dst_of(t, which, i));
        }
    };
    auto issue_k = [&](int t) { issue_any(kbase, p.ks.n, k_lane_off, t, 0); };
    auto issue_v = [&](int t) { issue_any(vbase, p.vs.n, v_lane_off, t, 1); };
    auto issue_full_kv = [&](int tk, int tv) {               // K tile tk and V tile tv, both full
        const uint16_t* ktile = kbase + (int64_t)tile_of(tk) * BN * p.ks.n;
        const uint16_t* vtile = vbase + (int64_t)tile_of(tv) * BN * p.vs.n;
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            dma16u(ktile, k_lane_off[i], dst_of(tk, 0, i));
            dma16u(vtile, v_lane_off[i], dst_of(tv, 1, i));
        }
    };
    // the first tiles are on their way before anything else is loaded: on short walks their round trip is the run time
#pragma unroll
    for (int i = 0; i < KD; ++i) {
        if (i < n_tiles) issue_k(i);
        if (i < VD && i < n_tiles) issue_v(i);
    }

    // ---- Q fragments (B operand of S^T = K Q^T): column = query, 8 consecutive d; through the place of V(1), or behind the stages
    bf16x8 qf[DC];
    {
        static_assert(T::q_pass_bytes(NW) == 0 || (KG == 1 && !BIAS && !KEYS), "nothing else lies behind the stages");
        u32x4 w[DC];
        load_rows32<D>(w, qbase + (int64_t)qw0 * p.qs.n, p.qs.n, p.Sq - qw0, p.d);
        fragments_of_rows32<D>(lds + (T::q_pass_bytes(NW) ? 2 * T::STAGE_ELEMS : T::STAGE_ELEMS + T::TILE_ELEMS) + wave * 1024, w,
                               [&](auto dc, u32x4 f) { qf[decltype(dc)::value] = __builtin_bit_cast(bf16x8, f); });
    }

    // ---- per-lane LDS read offsets (elements), constant over the key loop
    int koff[DC];          // K fragment: row 32*kb + n, logical granule 2*dc + h
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) koff[dc] = n * RS + (((2 * dc + h) ^ swz<D>(n)) << 3);
    const int tr_r = lane & 15, tr_g16 = (lane >> 4) & 1;
    int voff[2][DB];       // V^T fragment halves: rows 4h + r/4 (+8), logical granule 4*db + 2*g16 + (r&3)/2
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int row = 4 * h + (tr_r >> 2) + 8 * half;
#pragma unroll
        for (int db = 0; db < DB; ++db)
            voff[half][db] = row * RS + (((4 * db + 2 * tr_g16 + ((tr_r & 3) >> 1)) ^ swz<D>(row)) << 3) + 4 * (tr_r & 1);
    }
    auto k_frag = [&](int t, int i) {       // fragment i = (dc, kb) of K(t)
        const uint16_t* ks = lds + (t & 1) * T::STAGE_ELEMS;
        return *reinterpret_cast<const bf16x8*>(ks + koff[i >> 1] + 32 * (i & 1) * RS);
    };
    auto v_frag = [&](int t, int i) {       // fragment i = (cc, db) of V(t)^T
        const uint16_t* vs = lds + (t & 1) * T::STAGE_ELEMS + T::TILE_ELEMS;
        const int cc = i / DB, db = i % DB;
        const u32x2 lo = lds_read_tr16(vs + voff[0][db] + 16 * cc * RS);
        const u32x2 hi = lds_read_tr16(vs + voff[1][db] + 16 * cc * RS);
        const u32x4 u = {lo[0], lo[1], hi[0], hi[1]};
        return __builtin_bit_cast(bf16x8, u);
    };

    // ---- running state; each lane serves query column n
    const float c_log2 = p.scale * kLog2e;
    const float stale_ok = 8.0f / c_log2;     // the reference maximum may lag the true one by 2^8
    float m_run = -INFINITY, l_run = 0.f;
    f32x16 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;

    constexpr int NS = 2 * DC;     // logit MFMAs per tile
    constexpr int NP = 4 * DB;     // PV MFMAs per tile
    // logits 32 j / NS to 32 (j + 1) / NS belong to softmax slice j, pairs 16 i / NP to 16 (i + 1) / NP to maximum-scan slice i
    constexpr int EPS = (32 + NS - 1) / NS, PPS = (16 + NP - 1) / NP;

    // DROP: flat index (mod 2^32) of this lane's first element of the row in the [B*H, Sq, Sk] probability tensor
    const uint32_t drop_row = ((uint32_t)bh * (uint32_t)p.Sq + (uint32_t)qi) * (uint32_t)p.Sk + (uint32_t)key0 + 4 * h;
    (void)drop_row;
    // Exclusions of a tile.  The ragged tail / key length and the causal diagonal are one comparison per element with a
    // per-lane limit (excl_elem, threaded into the maximum scan); a keep-mask row is fetched when the step begins; the
    // general mask and bias are applied in one go (excl_general).
    int lim = 0;                   // keys of the tile below it attend, counted from 4h
    MaskRow64 mrow;
    uint32_t keep_bits[2];         // KEYS: of this lane's half, key block by key block
    // BITS: the word of the next cut tile.  Requested a step ahead: loads return in order, so that one which a step itself waits
    // for makes it wait for the copies that it has just issued as well.
    uint64_t word_ahead = 0;
    auto word_of = [&](int t) {
        return *reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(brows + (int64_t)kt.tile(t) * (64 * p.m.bit_nqt)) + 8u * (uint32_t)qi);
    };
    auto excl_begin = [&](int t) {
        if constexpr (KEYS) {
            const uint64_t w = BITS ? word_ahead : kt.bits[kt.tile(t)];
            if (BITS && t + 1 < n_tiles) word_ahead = word_of(t + 1);
            keep_bits[0] = (uint32_t)w >> (4 * h);
            keep_bits[1] = (uint32_t)(w >> 32) >> (4 * h);
        }
        const int limit = (p.m.causal ? min(klimit, qi + 1 - key0) : klimit) - t * BN;
        lim = limit - 4 * h;
        if constexpr (EXCL == kExRows16) {
            // folded into the mask bytes where they cut the tile: the per-element test is then the mask byte alone
            mrow.load(mbase + (int64_t)min(qi, p.Sq - 1) * p.m.sq + t * BN);
            if (__any(limit < BN)) mrow.restrict_to(limit);
        }
    };
    // Tiles below t_clean need no exclusions for any query of the workgroup; the rest (ragged tail, causal
    // diagonal, or everything under an explicit mask) carry per-element exclusions.
    int t_clean = KEYS ? kt.n_whole : (EXCL == kExNone || BIAS) ? klimit / BN : 0;
    if (p.m.causal) t_clean = min(t_clean, (q0 + 1 - key0) / BN);
    t_clean = max(min(t_clean, n_tiles), 0);
    if constexpr (BITS) {
        const int first = t_clean == 0 ? 0 : (t_clean - 1) | 1;      // that a step with exclusions takes: steps go in pairs, see below
        if (first < n_tiles) word_ahead = word_of(first);
    }

    // Bias: every lane needs 64 (of its half: 32) consecutive values of its query's row.  Four neighbouring lanes load 64 bytes
    // of a row (a "piece" is 16 rows of that, one instruction), and two pieces, 32 rows, at a time pass through 2 KiB of LDS
    // to the lanes that own the rows, granules swizzled as in fragments_of_rows32: an instruction whose lanes each load from
    // a row of their own keeps the address unit busy for 64 clocks instead of 16.  The pieces of the next tile are requested
    // across the logit phase, when the exponentials have freed the registers they take; a pair of them goes through LDS in
    // the PV phase, one ahead of the slices that add it.
    // (B=1 H=64 S=512 D=64, fp32: 84 MB move, 16 us at the rate of a copy; four values per lane and load 23.5 us, this 19.4.
    // B=3 H=16 S=1664 fp32: D = 64 123 -> 82 us, D = 128 166 -> 150 us; its two wavefronts per SIMD wait for the bias then.)
    // EARLY (D = 64, which has the registers): a pair of pieces is requested for the tile after the next as soon as it has gone through
    // LDS, so that it has a whole step to arrive instead of half of one, and the last wait of a step that
    // copies two whole tiles counts these loads out; the other steps request it behind their barrier, all at once.  A ragged tile is
    // requested across the logit phase as above.  B=1 H=64 S=512 19.7 -> 15.5 us, the rate of a copy; S=256 10.9 -> 8.0; B=1 H=12
    // S=2048 42.3 -> 36.6, B=4 H=64 S=700 84.7 -> 77.4, B=3 H=16 S=1664 78.5 -> 70.2 us; B=4 H=16 S=1344 gains
    // nothing (63.9 -> 65 us, and 59.8 to 60.8 over later runs).
    using BiasPiece = typename std::conditional<EXCL == kExBiasF32, f32x4_any, u16x8_any>::type;
    using BiasElem = typename std::conditional<EXCL == kExBiasF32, float, uint16_t>::type;
    constexpr int BEL = EXCL == kExBiasF32 ? 4 : 8;           // values per piece and lane
    constexpr int NPIECE = BIAS ? 32 / BEL : 1, NPASS = BIAS ? NPIECE / 2 : 1;
    constexpr bool EARLY = BIAS && AHEAD;
    BiasPiece bw[NPIECE];
    f32x4 bg[EXCL == kExBiasF32 ? 8 : 1];                     // keys 8 j + 4 h .. + 3 of this lane's row
    u32x2 bgh[EXCL == kExBiasBf16 ? 8 : 1];
    // the wavefront's first row, and this lane's place (bytes) in rows lane / 4 and lane / 4 + 16 (row pitches below 2^24 elements)
    const BiasElem* const brow0 = BIAS ? static_cast<const BiasElem*>(p.m.bias) + b * p.m.bb + hh * p.m.bh + (int64_t)min(qw0, p.Sq - 1) * p.m.bq : nullptr;
    uint32_t boff[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
        boff[u] = (uint32_t)sizeof(BiasElem) * (uint32_t)(min(16 * u + (lane >> 2), max(p.Sq - 1 - qw0, 0)) * (int)p.m.bq + BEL * (lane & 3));
    uint16_t* const bpass = lds + T::LDS_BYTES / 2 + wave * 1024;
    const int bto = (lane >> 2) * 32 + (((lane & 3) ^ ((lane >> 4) & 3)) << 3);
    const int bfrom = n * 32 + (EXCL == kExBiasF32 ? (h ^ ((n >> 2) & 3)) << 3 : (((n >> 2) & 3) << 3) + 4 * h);
    auto bias_request = [&](auto ragged_tag, int t, int i) {
        if constexpr (BIAS) {
            const int key = t * BN + 4 * BEL * (i >> 1);             // of lanes with lane % 4 == 0
            if constexpr (!decltype(ragged_tag)::value) {
                bw[i] = *reinterpret_cast<const BiasPiece*>(reinterpret_cast<const char*>(brow0 + key) + boff[i & 1]);
            } else {                                 // ragged tail: nothing past the row is read, keys past the end get -inf
                const BiasElem* row = reinterpret_cast<const BiasElem*>(reinterpret_cast<const char*>(brow0) + boff[i & 1]);
                const int last = p.Sk - 1 - BEL * (lane & 3);
#pragma unroll
                for (int e = 0; e < BEL; ++e) {
                    const BiasElem v = row[min(key + e, last)];
                    bw[i][e] = key + e > last ? (EXCL == kExBiasF32 ? (BiasElem)-INFINITY : (BiasElem)0xff80u) : v;
                }
            }
        }
    };
    auto bias_pass = [&](int c) {                    // pieces 2 c and 2 c + 1 to the rows' lanes
        if constexpr (BIAS) {
            *reinterpret_cast<u32x4*>(bpass + bto) = __builtin_bit_cast(u32x4, bw[2 * c]);
            *reinterpret_cast<u32x4*>(bpass + bto + 16 * 32) = __builtin_bit_cast(u32x4, bw[2 * c + 1]);
            if constexpr (EXCL == kExBiasF32) {      // granule 2 u + h
#pragma unroll
                for (int u = 0; u < 2; ++u) bg[2 * c + u] = *reinterpret_cast<const f32x4*>(bpass + (bfrom ^ (16 * u)));
            } else {                                 // half h of granule u
#pragma unroll
                for (int u = 0; u < 4; ++u) bgh[4 * c + u] = *reinterpret_cast<const u32x2*>(bpass + (bfrom ^ (8 * u)));
            }
        }
    };
    auto bias_request_whole = [&](int t) {
        if (t < t_clean) {
#pragma unroll
            for (int i = 0; i < NPIECE; ++i) bias_request(std::false_type{}, t, i);
        }
    };
    auto excl_elem = [&](f32x16 (&s)[2], int idx) {
        const int kb = idx >> 4, r = idx & 15;
        if constexpr (BIAS) {     // scale * (s + bias / scale) = scale * s + bias
            float v;
            if constexpr (EXCL == kExBiasF32) v = bg[idx >> 2][idx & 3];
            else v = idx & 1 ? bf16_hi(bgh[idx >> 2][(idx >> 1) & 1]) : bf16_lo(bgh[idx >> 2][(idx >> 1) & 1]);
            s[kb][r] = fmaf(v, p.m.inv_scale, s[kb][r]);
        }
        if constexpr (KEYS) s[kb][r] = keep_bits[kb] & (1u << (8 * (r >> 2) + (r & 3))) ? s[kb][r] : -INFINITY;
        if constexpr (EXCL == kExRows16) s[kb][r] = mrow.keep(kb, r, h) ? s[kb][r] : -INFINITY;
        if constexpr (EXCL == kExNone) s[kb][r] = 32 * kb + 8 * (r >> 2) + (r & 3) >= lim ? -INFINITY : s[kb][r];
    };
    auto excl_general = [&](f32x16 (&s)[2], int t) {
        // a lane's 64 keep-mask bytes of the tile in four 16-byte loads where the layout allows it (each
        // lane owns a query row, so byte loads would touch one cache line per lane and element)
        const bool vec_mask = mbase && p.m.rows16 && t * BN + BN <= p.Sk;
        if (vec_mask) mrow.load(mbase + (int64_t)min(qi, p.Sq - 1) * p.m.sq + t * BN);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = t * BN + 32 * kb + acc_row(r, h);
                bool drop = (key >= klimit) | ((p.m.causal != 0) & (key > qi));     // bitwise: selects, not branches
                float val = s[kb][r];
                if (vec_mask) drop = drop || !mrow.keep(kb, r, h);
                else if (mbase && !drop && qi < p.Sq) drop = !mask_attends(p.m, mbase, (int64_t)qi * p.m.sq + (int64_t)key * p.m.sk);
                if (bbase) {      // scale * (s + bias / scale) = scale * s + bias
                    float bv = 0.f;
                    if (!drop && qi < p.Sq) {
                        const int64_t e = (int64_t)qi * p.m.bq + (int64_t)key * p.m.bk;
                        bv = p.m.bias_f32 ? reinterpret_cast<const float*>(bbase)[e]
                                          : __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(bbase)[e] << 16);
                    }
                    val = fmaf(bv, p.m.inv_scale, val);
                }
                s[kb][r] = drop ? -INFINITY : val;   // select, not a divergent store
            }
    };
    // Fold the maximum of a freshly computed tile into the running state.  The reference maximum
    // moves (and the running sums are rescaled) only when some lane's tile maximum exceeds it by more
    // than 2^8 in the exponent domain; the branch is wave-uniform.  Both lanes of a query hold the same reference maximum, so
    // each may test its own half of the keys: the exchange between the halves stays inside the branch.
    auto fold_max = [&](float tmax) {
        if (__any(tmax > m_run + stale_ok)) {
            tmax = fmaxf(tmax, xhalf(tmax));
            const float m_old = m_run;
            const float m_new = fmaxf(m_old, tmax);
            const float m_to = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = exp2_fast((m_old - m_to) * c_log2);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
        }
    };
    auto zero_tile = [&](f32x16 (&s)[2]) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
    };

    // One step: P(t) from the logits in `cur`, logits of tile t+1 into `nxt`, O += P(t) V(t).
    // COPY: K(t+KD) and V(t+VD) exist and are full tiles (straight-line copies); else decided at run time.
    // NEXT: 0 = tile t+1 needs no exclusions, 1 = it does, 2 = tile t is the last one.
    auto step = [&](auto copy_tag, auto next_tag, f32x16 (&cur)[2], f32x16 (&nxt)[2], int t) {
        constexpr bool COPY = decltype(copy_tag)::value;
        constexpr int NEXT = decltype(next_tag)::value;
        if constexpr (COPY) {
            issue_full_kv(t + KD, t + VD);
        } else if constexpr (NEXT != 2) {
            if (t + KD < n_tiles) issue_k(t + KD);
            if (t + VD < n_tiles) issue_v(t + VD);
        }
        const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
        const float msc = m_use * c_log2;
        float rsum0 = 0.f, rsum1 = 0.f;
        bf16x8 pf[4];
        bf16x8 fb[PD];
        const uint32_t drop_tile = drop_row + (uint32_t)(t * BN), drop_word = DROP == kDropRows64 ? xorshift32(p.m.drop_seed ^ drop_tile) : 0u;
        (void)drop_tile;
        (void)drop_word;
        // P(t): the logits of the tile in (kb, r) order
        auto exp_slice = [&](int j) {
#pragma unroll
            for (int e = 0; e < EPS; ++e) {
                const int idx = 32 * j / NS + e, kb = idx >> 4, r = idx & 15;
                if (idx >= 32 * (j + 1) / NS) continue;
                const float v = exp2_fast(fmaf(cur[kb][r], c_log2, -msc));
                if (idx & 1) rsum1 += v;
                else rsum0 += v;
                const uint32_t off = 32 * kb + 8 * (r >> 2) + (r & 3);       // of the element, from drop_tile
                if constexpr (DROP == kDropTiled) {
                    cur[kb][r] = v * drop_factor_at(p.m, (uint32_t)bh, (uint32_t)qi, (uint32_t)(key0 + t * BN + 4 * h) + off, (uint32_t)p.Sq, (uint32_t)p.Sk);
                } else if constexpr (DROP != kDropNone) {
                    const uint32_t w = DROP == kDropRows64 ? drop_word ^ xorshift32(off) : xorshift32(p.m.drop_seed ^ (drop_tile + off));
                    cur[kb][r] = w >= p.m.drop_thr32 ? v : 0.f;
                } else {
                    cur[kb][r] = v;
                }
                if ((idx & 7) == 7) {
                    const int o8 = r - 7;
                    const f32x16& s = cur[kb];
                    pf[idx >> 3] = pack8(s[o8 + 0], s[o8 + 1], s[o8 + 2], s[o8 + 3], s[o8 + 4], s[o8 + 5], s[o8 + 6], s[o8 + 7]);
                }
            }
        };
        if constexpr (NEXT == 2) {
#pragma unroll
            for (int i = 0; i < PD; ++i) {
                fb[i] = v_frag(t, i);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < NS; ++j) exp_slice(j);
            l_run += rsum0 + rsum1;
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                oacc[i % DB] = mfma32(fb[i % PD], pf[i / DB], oacc[i % DB]);
                if (i + PD < NP) fb[i % PD] = v_frag(t, i + PD);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            if (NEXT == 1) excl_begin(t + 1);
            const std::integral_constant<bool, NEXT == 1> ragged_tag{};
            // ---- S(t+1)^T = K(t+1) Q^T between the exponentials of tile t
            zero_tile(nxt);
#pragma unroll
            for (int i = 0; i < PD; ++i) {
                fb[i] = k_frag(t + 1, i);
                __builtin_amdgcn_sched_barrier(0);
            }
            // Fragments are consumed in pairs, the younger read of a pair first: LDS returns in order, so
            // the wait for it also covers its partner and one s_waitcnt serves two MFMAs.  The two reads
            // that refill the ring are issued together at the end of the pair.
            auto frag_of = [&](int f) { return f < NS ? k_frag(t + 1, f) : v_frag(t, f - NS); };   // f in [0, NS + NP)
#pragma unroll
            for (int i = 0; i < NS; i += 2) {
                nxt[1] = mfma32(fb[(i + 1) % PD], qf[i >> 1], nxt[1]);
                exp_slice(i);
                if (BIAS && (!EARLY || (NEXT == 1 && t + 1 >= t_clean)) && i % (NS / NPIECE) == 0) bias_request(ragged_tag, t + 1, i / (NS / NPIECE));
                __builtin_amdgcn_sched_barrier(0);
                nxt[0] = mfma32(fb[i % PD], qf[i >> 1], nxt[0]);
                exp_slice(i + 1);
                if (BIAS && (!EARLY || (NEXT == 1 && t + 1 >= t_clean)) && (i + 1) % (NS / NPIECE) == 0) bias_request(ragged_tag, t + 1, (i + 1) / (NS / NPIECE));
                fb[i % PD] = frag_of(i + PD);
                fb[(i + 1) % PD] = frag_of(i + 1 + PD);
                __builtin_amdgcn_sched_barrier(0);
            }
            l_run += rsum0 + rsum1;
            if (NEXT == 1 && EXCL == kExGeneral) excl_general(nxt, t + 1);
            // ---- O^T += V(t)^T P(t)^T between the row-maximum scan of tile t+1
            float tmax = -INFINITY;
            auto bias_through = [&](int c) {
                bias_pass(c);
                if (EARLY && COPY) {       // tile t + 2 is a whole one
                    bias_request(std::false_type{}, t + 2, 2 * c);
                    bias_request(std::false_type{}, t + 2, 2 * c + 1);
                }
            };
            if constexpr (BIAS) bias_through(0);
            auto max_slice = [&](int i) {
                if (BIAS && i % (NP / NPASS) == 0 && i / (NP / NPASS) + 1 < NPASS) bias_through(i / (NP / NPASS) + 1);
#pragma unroll
                for (int e = 0; e < PPS; ++e) {
                    const int idx = 2 * (16 * i / NP + e);
                    if (idx >= 2 * (16 * (i + 1) / NP)) continue;
                    if (NEXT == 1 || BIAS) {
                        excl_elem(nxt, idx);
                        excl_elem(nxt, idx + 1);
                    }
                    tmax = fmaxf(fmaxf(tmax, nxt[idx >> 4][idx & 15]), nxt[(idx + 1) >> 4][(idx + 1) & 15]);
                }
            };
#pragma unroll
            for (int i = 0; i < NP; i += 2) {
                oacc[(i + 1) % DB] = mfma32(fb[(i + 1) % PD], pf[(i + 1) / DB], oacc[(i + 1) % DB]);
                max_slice(i);
                __builtin_amdgcn_sched_barrier(0);
                oacc[i % DB] = mfma32(fb[i % PD], pf[i / DB], oacc[i % DB]);
                max_slice(i + 1);
                if (i + PD < NP) {
                    fb[i % PD] = frag_of(NS + i + PD);
                    fb[(i + 1) % PD] = frag_of(NS + i + 1 + PD);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            fold_max(tmax);
            // the copies issued by this step have landed
            if constexpr (EARLY && COPY) wait_vm<NPIECE>();          // (younger than they are: the bias of tile t + 2)
            else wait_vm0();
            __syncthreads();     // ... for every wave, and everyone is done reading this step's tiles
            if constexpr (EARLY && !COPY) bias_request_whole(t + 2);
        }
    };

    f32x16 sa[2], sb[2];
    if (n_tiles > 0) {
        wait_vm0();
        __syncthreads();
        if (t_clean == 0) excl_begin(0);
        if constexpr (BIAS) {
            if (t_clean > 0) {
#pragma unroll
                for (int i = 0; i < NPIECE; ++i) bias_request(std::false_type{}, 0, i);
            } else {
#pragma unroll
                for (int i = 0; i < NPIECE; ++i) bias_request(std::true_type{}, 0, i);
            }
        }
        zero_tile(sa);
#pragma unroll
        for (int i = 0; i < NS; ++i) sa[i & 1] = mfma32(k_frag(0, i), qf[i >> 1], sa[i & 1]);
        if (t_clean == 0 || BIAS) {
            if (EXCL == kExGeneral) excl_general(sa, 0);
            if constexpr (BIAS) {
#pragma unroll
                for (int c = 0; c < NPASS; ++c) bias_pass(c);
            }
#pragma unroll
            for (int idx = 0; idx < 32; ++idx) excl_elem(sa, idx);
        }
        if constexpr (EARLY) bias_request_whole(1);
        float tmax = sa[0][0];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sa[kb][r]);
        fold_max(tmax);
        __syncthreads();     // every wave has read K(0) before step 0 starts overwriting it

        using Yes = std::true_type;
        using No = std::false_type;
        using Clean = std::integral_constant<int, 0>;
        using Cut = std::integral_constant<int, 1>;
        using Last = std::integral_constant<int, 2>;
        // Two steps per trip, so that `sa` is the current tile when t is even; where the number of steps of
        // one kind is odd, the pair that mixes kinds runs as the more general one.
        int t = 0;
        if (EXCL == kExNone || BIAS || KEYS) {
            const int copy_end = t_clean - KD;              // steps below it copy two full tiles
            for (; t + 1 < copy_end; t += 2) {
                step(Yes{}, Clean{}, sa, sb, t);
                step(Yes{}, Clean{}, sb, sa, t + 1);
            }
            for (; t + 2 < t_clean; t += 2) {
                step(No{}, Clean{}, sa, sb, t);
                step(No{}, Clean{}, sb, sa, t + 1);
            }
        }
        if (EXCL == kExRows16 || EXCL == kExGeneral) {
            const int copy_end = min(n_tiles, klimit / BN) - KD;
            for (; t + 1 < copy_end; t += 2) {
                step(Yes{}, Cut{}, sa, sb, t);
                step(Yes{}, Cut{}, sb, sa, t + 1);
            }
        }
        for (; t + 2 < n_tiles; t += 2) {
            step(No{}, Cut{}, sa, sb, t);
            step(No{}, Cut{}, sb, sa, t + 1);
        }
        if (t + 1 < n_tiles) {
            step(No{}, Cut{}, sa, sb, t);
            step(No{}, Last{}, sb, sa, t + 1);
        } else {
            step(No{}, Last{}, sa, sb, t);
        }
    }

    // ---- the second group's state joins the first's
    if constexpr (KG == 2) {
        // a walk of n tiles passes n + 1 barriers; the second group's may be one tile shorter, or empty
        const int mine = n_tiles > 0 ? n_tiles + 1 : 0, most = n_first > 0 ? n_first + 1 : 0;
        for (int i = mine; i < most; ++i) __syncthreads();
        __syncthreads();                               // nobody reads a tile any more
        static_assert(NW * (4 * DB + 1) * 64 * 16 <= KG * T::LDS_BYTES, "the state of a group fits where the tiles were");
        f32x4* slot = reinterpret_cast<f32x4*>(lds_all) + wave * (4 * DB + 1) * 64 + lane;
        if (group == 1) {
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i) {
                const f32x16& a = oacc[i >> 2];
                slot[64 * i] = f32x4{a[4 * (i & 3)], a[4 * (i & 3) + 1], a[4 * (i & 3) + 2], a[4 * (i & 3) + 3]};
            }
            slot[64 * 4 * DB] = f32x4{m_run, l_run, 0.f, 0.f};
        }
        __syncthreads();
        if (group == 1) return;
        const f32x4 other = slot[64 * 4 * DB];
        const float m_new = fmaxf(m_run, other[0]), m_to = (m_new == -INFINITY) ? 0.f : m_new;
        const float w0 = exp2_fast((m_run - m_to) * c_log2), w1 = exp2_fast((other[0] - m_to) * c_log2);
        l_run = l_run * w0 + other[1] * w1;
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < 4 * DB; ++i) {
            const f32x4 v = slot[64 * i];
#pragma unroll
            for (int e = 0; e < 4; ++e) oacc[i >> 2][4 * (i & 3) + e] = fmaf(oacc[i >> 2][4 * (i & 3) + e], w0, v[e] * w1);
        }
    }

    // ---- epilogue: O through LDS where nobody reads any more (KG: the state of the second group this wavefront has joined)
    if constexpr (KG == 1) __syncthreads();
    uint16_t* own = KG == 1 ? lds + wave * 32 * RS : lds_all + wave * (4 * DB + 1) * 64 * 8;
    const float l = l_run + xhalf(l_run);
    float inv = l > 0.f ? 1.0f / l : 0.f;
    if constexpr (DROP == kDropFlat || DROP == kDropRows64) inv *= p.m.drop_scale;
    store_rows32<D>(own, p.o + b * p.os.b + hh * p.os.h + (int64_t)qw0 * p.os.n, p.os.n, p.Sq - qw0, p.dv, [&](int db, int g) {
        const f32x16& a = oacc[db];
        return u32x2{pack_bf16(a[4 * g] * inv, a[4 * g + 1] * inv), pack_bf16(a[4 * g + 2] * inv, a[4 * g + 3] * inv)};
    });
    if (p.lse && h == 0 && qi < p.Sq) p.lse[(int64_t)bh * p.Sq + qi] = l > 0.f ? (m_run * c_log2 + log2_fast(l)) * kLn2 : -INFINITY;
}

template <int D, int EXCL, int NW, int DROP = kDropNone, int KG = 1, bool AHEAD = false>
__global__ __launch_bounds__(64 * NW * KG, NW * KG == 4 || KG == 2 ? 2 : 1) void fwd_kernel(const FwdParams p) {
    fwd_body<D, EXCL, NW, DROP, KG, AHEAD, false>(p);
}
template <int D, int EXCL, int NW>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void fwd_dealt_kernel(const FwdParams p) {
    fwd_body<D, EXCL, NW, kDropNone, 1, false, true>(p);
}

// Combines the partial outputs of a key split: LSE = log sum_s exp(LSE_s), O = sum_s exp(LSE_s - LSE) O_s.  A slice whose sum
// was NaN makes O NaN (and LSE -inf, as in a walk over all keys by one workgroup).  One lane per query row and 4 output columns.
static __global__ __launch_bounds__(256) void fwd_merge_kernel(const FwdParams p) {
    const int groups = p.dv >> 2;
    const int64_t rows = (int64_t)p.B * p.H * p.Sq;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * groups) return;
    const int64_t row = idx / groups;
    const int g = (int)(idx % groups);
    float m = -INFINITY;
    bool nan = false;                  // fmaxf passes over a NaN
    for (int s = 0; s < p.key_splits; ++s) {
        const float l = p.part_lse[s * rows + row];
        m = fmaxf(m, l);
        nan |= l != l;
    }
    float sum = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (m != -INFINITY || nan) {
        for (int s = 0; s < p.key_splits; ++s) {
            const float w = expf(p.part_lse[s * rows + row] - m);
            const f32x4 v = *reinterpret_cast<const f32x4*>(p.part_o + (s * rows + row) * p.dv + 4 * g);
            sum += w;
            acc[0] = fmaf(w, v[0], acc[0]); acc[1] = fmaf(w, v[1], acc[1]);
            acc[2] = fmaf(w, v[2], acc[2]); acc[3] = fmaf(w, v[3], acc[3]);
        }
    }
    const float inv = sum > 0.f ? 1.0f / sum : 0.f;
    const int64_t bh = row / p.Sq, qi = row % p.Sq;
    uint16_t* orow = p.o + (bh / p.H) * p.os.b + (bh % p.H) * p.os.h + qi * p.os.n;
    const u32x2 w = {pack_bf16(acc[0] * inv, acc[1] * inv), pack_bf16(acc[2] * inv, acc[3] * inv)};
    *reinterpret_cast<u32x2*>(orow + 4 * g) = w;
    if (p.lse && g == 0) p.lse[row] = sum > 0.f ? m + logf(sum) : -INFINITY;
}

// ------------------------------------------------------------------- forward, 256-query workgroups
// The same computation as fwd_kernel for workgroups of 256 queries, laid out for one wavefront per
// SIMD: 4 wavefronts of 64 queries (two 32-query blocks) each, so that every K / V fragment read from
// LDS feeds two MFMAs and the LDS reads and waits per MFMA halve.  O^T of both blocks and the Q
// fragments live in the accumulation registers (Q as pinned MFMA B operands), the logits in
// architectural registers through hand-emitted MFMAs (see mfma32_vgpr_bacc): nothing may touch them until
// two further MFMAs have been issued.  Four LDS stages, K(t) and V(t) in stage t % 4: step t reads
// K(t+1) and V(t) and issues the copies of K(t+3) and V(t+2), each into a slot whose previous tile was
// last read two barriers ago, and each with more than a full step to land; one workgroup barrier
// per step, placed just before the fragment ring first reads K(t+2); the ring runs on across steps.
// Every step is the pipelined one: the kernel serves problems without any exclusion (no causal
// flag, key lengths, keep-mask or bias, Sk a multiple of 64); all others use fwd_kernel.  Copies past the
// last tile re-read the last tile, and the logits "of the tile after the last" are never used.  A
// kernel of this size must not spill: scratch memory per wavefront limits how many workgroups the
// device keeps resident, which halved the throughput of a version with a general slow path.
template <int D>
struct FwdWideTile {
    static constexpr int BM = 256;
    static constexpr int BN = 64;
    static constexpr int RS = kRowPitch<D>;
    static constexpr int TILE_ELEMS = BN * RS;
    static constexpr int STAGE_ELEMS = 2 * TILE_ELEMS;
    static constexpr int NSTAGE = 4;
    static constexpr int LDS_BYTES = NSTAGE * STAGE_ELEMS * 2;
    static constexpr int ROWS_PER_DMA = 1024 / (RS * 2);
    static constexpr int DMA_PER_WAVE = BN / ROWS_PER_DMA / 4;
};

template <int D>
__global__ __launch_bounds__(256) void fwd_wide_kernel(const FwdParams p) {
    using T = FwdWideTile<D>;
    constexpr int BN = T::BN, RS = T::RS, BM = T::BM;
    constexpr int DC = D / 16, DB = D / 32, GPR = RS / 8;
    constexpr int NDMA = T::DMA_PER_WAVE;
    constexpr int PD = 4;
    constexpr int NKF = 2 * DC;          // K fragments per tile (dc, kb); two logit MFMAs each
    constexpr int NVF = 4 * DB;          // V^T fragments per tile (16-key chunk, db); two PV MFMAs each
    static_assert(NKF % PD == 0 && NVF % PD == 0, "read-ahead depth must divide the fragment counts");
    static_assert(DB <= 4, "O^T tuples are pinned four to a query block");

    extern __shared__ __attribute__((aligned(1024))) uint16_t lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;

    const int n_qt = (p.Sq + BM - 1) / BM;
    const int wg = xcd_remap(blockIdx.x, gridDim.x);
    const int qt = wg % n_qt;
    const int bh = wg / n_qt;
    const int b = bh / p.H, hh = bh % p.H;
    const int q0 = qt * BM;
    const int qw0 = q0 + wave * 64;

    const uint16_t* qbase = p.q + b * p.qs.b + hh * p.qs.h;
    const uint16_t* kbase = p.k + b * p.ks.b + hh * p.ks.h;
    const uint16_t* vbase = p.v + b * p.vs.b + hh * p.vs.h;
    uint16_t* obase = p.o + b * p.os.b + hh * p.os.h;

    const int n_tiles = p.Sk / BN;          // the launcher guarantees Sk % BN == 0 and no exclusions

    // ---- asynchronous tile copies: tile t (K and V) lives in stage t % 4
    const uint32_t lds0 = lds_addr(lds);
    const int dma_row_in = lane / GPR, dma_gran = lane % GPR;
    uint32_t k_lane_off[NDMA], v_lane_off[NDMA];
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int row = (wave * NDMA + i) * T::ROWS_PER_DMA + dma_row_in;
        const int c = dma_gran ^ swz<D>(row);
        k_lane_off[i] = 2u * (uint32_t)(row * (int)p.ks.n + src_granule(c, p.d) * 8);
        v_lane_off[i] = 2u * (uint32_t)(row * (int)p.vs.n + src_granule(c, p.dv) * 8);
    }
    auto dst_of = [&](int stg, int which, int i) {
        return lds0 + 2u * (uint32_t)(stg * T::STAGE_ELEMS + which * T::TILE_ELEMS + (wave * NDMA + i) * 512);
    };
    // whole tile t (clamped to the last one) of K or V into stage t % 4, all copies at once (prologue)
    auto issue_whole = [&](const uint16_t* base, int64_t row_stride, const uint32_t (&lane_off)[NDMA], int t, int which) {
        const uint16_t* tb = base + (int64_t)min(t, n_tiles - 1) * BN * row_stride;
#pragma unroll
        for (int i = 0; i < NDMA; ++i) dma16u(tb, lane_off[i], dst_of(t & 3, which, i));
    };
    // K(0) and Q first: the logits of the first tile need no more
    if (n_tiles > 0) issue_whole(kbase, p.ks.n, k_lane_off, 0, 0);

    // ---- Q fragments (B operand of S^T = K Q^T): column = query, 8 consecutive d; pinned slots qb*DC + dc; through stage 3
    bf16x8 qf[2][DC];
    int qrow[2];
    {
        u32x4 w[2][DC];
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            qrow[qb] = qw0 + 32 * qb + n;
            load_rows32<D>(w[qb], qbase + (int64_t)(qw0 + 32 * qb) * p.qs.n, p.qs.n, p.Sq - qw0 - 32 * qb, p.d);
        }
        static_for<2>([&](auto qb_tag) {
            constexpr int qb = decltype(qb_tag)::value;
            fragments_of_rows32<D>(lds + 3 * T::STAGE_ELEMS + wave * 1024, w[qb], [&](auto dc_tag, u32x4 f) {
                constexpr int dc = decltype(dc_tag)::value;
                qf[qb][dc] = pin_b_fragment<qb * DC + dc>(f);
            });
        });
    }

    // ---- per-lane LDS read offsets (elements), constant over the key loop
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
    auto k_frag = [&](const uint16_t* stage, int i) {       // fragment i = (dc, kb)
        return *reinterpret_cast<const bf16x8*>(stage + koff[i >> 1] + 32 * (i & 1) * RS);
    };
    auto v_frag = [&](const uint16_t* stage, int i) {       // fragment i = (cc, db) of V^T
        const uint16_t* vs = stage + T::TILE_ELEMS;
        const int cc = i / DB, db = i % DB;
        const u32x2 lo = lds_read_tr16(vs + voff[0][db] + 16 * cc * RS);
        const u32x2 hi = lds_read_tr16(vs + voff[1][db] + 16 * cc * RS);
        const u32x4 u = {lo[0], lo[1], hi[0], hi[1]};
        return __builtin_bit_cast(bf16x8, u);
    };

    // ---- running state; each lane serves query column n of both blocks
    const float c_log2 = p.scale * kLog2e;
    const float stale_ok = 8.0f / c_log2;
    float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
    f32x16 oacc[2][DB];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[qb][db][r] = 0.f;

    // Fold the tile maximum of one query block into its running state (see fwd_kernel).  O^T of block
    // qb is pinned to a[64 qb : 64 qb + 63] for the rescale.
    auto fold_max = [&](auto qb_tag, float tmax) {
        constexpr int qb = decltype(qb_tag)::value;
        tmax = fmaxf(tmax, xhalf(tmax));
        if (__any(tmax > m_run[qb] + stale_ok)) {
            const float m_old = m_run[qb];
            const float m_new = fmaxf(m_old, tmax);
            const float m_to = (m_new == -INFINITY) ? 0.f : m_new;
            const float alpha = exp2_fast((m_old - m_to) * c_log2);
            m_run[qb] = m_new;
            l_run[qb] *= alpha;
            static_for<DB>([&](auto db_tag) {
                constexpr int db = decltype(db_tag)::value;
                rescale_pinned<4 * qb + db>(oacc[qb][db], alpha);
            });
        }
    };
    // the first tile: nothing accumulated yet
    auto first_max = [&](int qb, float tmax) { m_run[qb] = fmaxf(tmax, xhalf(tmax)); };
    // the hand-emitted MFMAs' results become visible 11 issue cycles after issue; the logits pass through
    // the statement so that nothing that reads them can be scheduled ahead of it
    auto settle = [&](f32x16 (&s)[2][2]) {
        asm volatile("s_nop 7\n\ts_nop 7" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]));
    };
    // S(t)^T of both query blocks from the K tile in `stage`, no overlap (prologue and slow steps)
    auto logits_plain = [&](f32x16 (&s)[2][2], const uint16_t* stage) {
        static_for<NKF>([&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            const bf16x8 kfr = k_frag(stage, i);
            static_for<2>([&](auto qb_tag) {
                constexpr int qb = decltype(qb_tag)::value;
                mfma32_vgpr_bpinned<qb * DC + (i >> 1), (i >> 1) == 0 ? 0 : 1>(s[qb][i & 1], kfr, qf[qb][i >> 1], s[qb][i & 1]);
            });
        });
        settle(s);
    };
    auto tile_max = [&](const f32x16 (&s)[2]) {
        float tmax = s[0][0];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[kb][r]);
        return tmax;
    };

    bf16x8 fb[PD];
    // One step: P(t) from the logits in `cur`, logits of tile t+1 into `nxt`, O += P(t) V(t).  MFMA slot
    // = 2 * fragment + query block.  The exponentials of the first key block of tile t are threaded between
    // the logit MFMAs of tile t+1; those of the second key block (needed from the middle of the PV products
    // on) between the first half of the MFMAs of O += P(t) V(t), the row-maximum scan of tile t+1 between
    // the second half: the wavefront is bound by instruction issue, so every slot gets its share.
    // STAGE: stage of tile t (0 .. 3).  k3_base / v2_base: tiles t+3 of K and t+2 of V (clamped).
    auto step = [&](auto stage_tag, f32x16 (&cur)[2][2], f32x16 (&nxt)[2][2], const uint16_t* k3_base,
                    const uint16_t* v2_base) {
        constexpr int s0 = decltype(stage_tag)::value;
        constexpr int s1 = (s0 + 1) & 3, s2 = (s0 + 2) & 3, s3 = (s0 + 3) & 3;
        const uint16_t* stage_t = lds + s0 * T::STAGE_ELEMS;       // V(t)
        const uint16_t* stage_t1 = lds + s1 * T::STAGE_ELEMS;      // K(t+1)
        const uint16_t* stage_t2 = lds + s2 * T::STAGE_ELEMS;      // K(t+2), landed during this step at the latest
        float msc[2], rsum0[2] = {0.f, 0.f}, rsum1[2] = {0.f, 0.f};
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) msc[qb] = ((m_run[qb] == -INFINITY) ? 0.f : m_run[qb]) * c_log2;
        u32x4 pw[2][4];                 // P^T operands: [query block][16-key chunk]
        // exponential of logit idx (in (kb, r) order) of query block qb
        auto exp_elem = [&](int qb, int idx) {
            const int kb = idx >> 4, r = idx & 15;
            cur[qb][kb][r] = exp2_fast(fmaf(cur[qb][kb][r], c_log2, -msc[qb]));
        };
        // Sums and packs a pair one slot after its exponentials, so that nothing waits on the transcendental
        // unit.  (The row sum is taken over the unrounded values: summing the packed pair with one
        // v_dot2_f32_bf16 would save an instruction per pair, but moves the logsumexp of a row that one key
        // dominates by up to 2^-9.)
        auto pack_pair = [&](int qb, int j) {
            const int idx = 2 * j, kb = idx >> 4, r = idx & 15;
            rsum0[qb] += cur[qb][kb][r];
            rsum1[qb] += cur[qb][kb][r + 1];
            pw[qb][idx >> 3][(idx & 7) >> 1] = pack_bf16(cur[qb][kb][r], cur[qb][kb][r + 1]);
        };

        {
            constexpr int NSL = 2 * NKF;             // MFMA slots of the logit phase
            // copies of K(t+3) and V(t+2); copy j goes with slot CS*j + 1
            constexpr int NCOPY = 2 * NDMA, CS = (NSL - 2) / NCOPY;
            // exponentials per slot and query block: the first key block's in the logit phase, the second's
            // in the first half of the other phase, whose slots have the vector unit to spare
            constexpr int HV = NVF / 2;
            constexpr auto e1 = [](int i) { return 16 * i / NKF; };        // the first of slot i
            constexpr auto e2 = [](int i) { return 16 * i / HV; };
            constexpr auto scan = [](int k) { return 32 * k / HV; };       // of the row maximum, in the second half
            static_assert(CS >= 2, "copies do not fit the logit phase");
            auto copy_dst = [&](int g) {
                const int j = (g - 1) / CS;
                if (g >= 1 && (g - 1) % CS == 0 && j < NCOPY) dma_set_dst(dst_of(j < NDMA ? s3 : s2, j / NDMA, j % NDMA));
            };
            auto copy_issue = [&](int g) {
                const int j = (g - 1) / CS;
                if (g >= 1 && (g - 1) % CS == 0 && j < NCOPY) {
                    if (j < NDMA) dma16u_issue(k3_base, k_lane_off[j]);
                    else dma16u_issue(v2_base, v_lane_off[j - NDMA]);
                }
            };
            // ---- S(t+1)^T = K(t+1) Q^T between the exponentials of tile t
            static_for<NKF>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                static_for<2>([&](auto qb_tag) {
                    constexpr int qb = decltype(qb_tag)::value;
                    constexpr int g = 2 * i + qb;
                    copy_dst(g);
                    if (qb == 0 && !(i & 1)) {
                        // one wait for the two fragments the ring read together; the pair read after them stays in flight
                        constexpr int younger = (i + 2 < NKF ? 1 : 2) + (i + 3 < NKF ? 1 : 2);
                        wait_lds_reads<younger>();
                    }
                    mfma32_vgpr_bpinned<qb * DC + (i >> 1), (i >> 1) == 0 ? 0 : 1>(nxt[qb][i & 1], fb[i % PD], qf[qb][i >> 1], nxt[qb][i & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                    copy_issue(g);
                    // slot g: exponentials of logits of the first key block of query block qb, packing of the pairs that
                    // were complete a slot ago
#pragma unroll
                    for (int e = e1(i); e < e1(i + 1); ++e) exp_elem(qb, e);
                    if (i > 0) {
#pragma unroll
                        for (int j = e1(i - 1) / 2; j < e1(i) / 2; ++j) pack_pair(qb, j);
                    }
                    // the ring is refilled two fragments at a time, so that one wait covers both
                    if (qb == 1 && (i & 1)) {
#pragma unroll
                        for (int f = i - 1; f <= i; ++f) {
                            if (f + PD < NKF) fb[f % PD] = k_frag(stage_t1, f + PD);
                            else fb[f % PD] = v_frag(stage_t, f + PD - NKF);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
#pragma unroll
                for (int j = e1(NKF - 1) / 2; j < 8; ++j) pack_pair(qb, j);
            }
            // ---- O^T += V(t)^T P(t)^T, with the rest of the exponentials and the row-maximum scan of tile t+1
            float tmax[2];
            static_for<NVF>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                constexpr int cc = i / DB, db = i % DB;
                static_for<2>([&](auto qb_tag) {
                    constexpr int qb = decltype(qb_tag)::value;
                    if (qb == 0 && !(i & 1)) {
                        constexpr int younger = (i + 2 < NVF ? 2 : 1) + (i + 3 < NVF ? 2 : 1);
                        wait_lds_reads<younger>();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    oacc[qb][db] = mfma32(fb[i % PD], __builtin_bit_cast(bf16x8, pw[qb][cc]), oacc[qb][db]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (i < HV) {
                        // first half: the exponentials of the second key block, due at slot HV
#pragma unroll
                        for (int e = e2(i); e < e2(i + 1); ++e) exp_elem(qb, 16 + e);
                    }
                    if (i >= 1 && i <= HV) {
#pragma unroll
                        for (int j = 8 + e2(i - 1) / 2; j < 8 + e2(i) / 2; ++j) pack_pair(qb, j);
                    }
                    if (i >= HV) {
                        // second half: row maximum of tile t+1 (its logits may be touched from slot 2 on)
                        constexpr int k = i - HV;
                        if (k == 0) tmax[qb] = nxt[qb][0][0];
#pragma unroll
                        for (int idx = scan(k); idx < scan(k + 1); ++idx) tmax[qb] = fmaxf(tmax[qb], nxt[qb][idx >> 4][idx & 15]);
                        // the scan feeds nothing before the end of the step: keep this slot's part in this slot
                        asm volatile("" : "+v"(tmax[qb]));
                    }
                    if (qb == 1) {
                        if (i == NVF - PD) {
                            __builtin_amdgcn_sched_barrier(0);
                            // the copies of the step before (K(t+2), V(t+1)) have landed; this step's may be in flight ...
                            __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * NDMA) & 15) | (((2 * NDMA) >> 4) << 14));
                            __builtin_amdgcn_s_barrier();    // ... for every wave, and every wave is past tile t-1
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        if (i & 1) {
#pragma unroll
                            for (int f = i - 1; f <= i; ++f) {
                                if (f + PD < NVF) fb[f % PD] = v_frag(stage_t, f + PD);
                                else fb[f % PD] = k_frag(stage_t2, f + PD - NVF);
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) l_run[qb] += rsum0[qb] + rsum1[qb];
            // Both lanes of a query hold the same reference maximum, so each may test its own half; the
            // exchange between the halves and the rescale stay inside the rarely taken branch.
            if (__any(tmax[0] > m_run[0] + stale_ok || tmax[1] > m_run[1] + stale_ok)) {
                fold_max(std::integral_constant<int, 0>{}, tmax[0]);
                fold_max(std::integral_constant<int, 1>{}, tmax[1]);
            }
        }
    };

    f32x16 sa[2][2], sb[2][2];
    if (n_tiles > 0) {
        // prologue: logits and maximum of tile 0 while K(1..2) and V(0..1) are on their way; the ring starts on K(1)
        wait_vm0();
        issue_whole(kbase, p.ks.n, k_lane_off, 1, 0);
        issue_whole(vbase, p.vs.n, v_lane_off, 0, 1);
        issue_whole(kbase, p.ks.n, k_lane_off, 2, 0);
        issue_whole(vbase, p.vs.n, v_lane_off, 1, 1);
        asm volatile("s_barrier" ::: "memory");        // K(0) has landed for every wave
        logits_plain(sa, lds);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) first_max(qb, tile_max(sa[qb]));
        wait_vm0();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PD; ++i) fb[i] = k_frag(lds + T::STAGE_ELEMS, i);

        const int64_t k_tile_stride = (int64_t)BN * p.ks.n, v_tile_stride = (int64_t)BN * p.vs.n;
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        // Tile t sits in stage t % 4 and its logits in `sa` when t is even: four step bodies.
        // K(t+3) and V(t+2) of the step at hand; copies past the last tile re-read the last tile
        const uint16_t* k3 = kbase + (int64_t)min(3, n_tiles - 1) * k_tile_stride;
        const uint16_t* v2 = vbase + (int64_t)min(2, n_tiles - 1) * v_tile_stride;
        auto advance = [&](int t) {    // from step t to step t+1
            k3 += (t + 4 < n_tiles) ? k_tile_stride : 0;
            v2 += (t + 3 < n_tiles) ? v_tile_stride : 0;
        };
        for (int t = 0; t < n_tiles; t += 4) {
            step(I0{}, sa, sb, k3, v2);
            if (t + 1 >= n_tiles) break;
            advance(t);
            step(I1{}, sb, sa, k3, v2);
            if (t + 2 >= n_tiles) break;
            advance(t + 1);
            step(I2{}, sa, sb, k3, v2);
            if (t + 3 >= n_tiles) break;
            advance(t + 2);
            step(I3{}, sb, sa, k3, v2);
            advance(t + 3);
        }
        wait_vm0();          // no copy may land where O passes through LDS
    }

    // ---- epilogue
    __syncthreads();
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int row = qrow[qb], row0 = qw0 + 32 * qb;
        const float l = l_run[qb] + xhalf(l_run[qb]);
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        store_rows32<D>(lds + wave * 32 * RS, obase + (int64_t)row0 * p.os.n, p.os.n, p.Sq - row0, p.dv, [&](int db, int g) {
            const f32x16& a = oacc[qb][db];
            return u32x2{pack_bf16(a[4 * g] * inv, a[4 * g + 1] * inv), pack_bf16(a[4 * g + 2] * inv, a[4 * g + 3] * inv)};
        });
        if (p.lse && h == 0 && row < p.Sq) p.lse[(int64_t)bh * p.Sq + row] = l > 0.f ? (m_run[qb] * c_log2 + log2_fast(l)) * kLn2 : -INFINITY;
    }
}

}  // namespace fattn
