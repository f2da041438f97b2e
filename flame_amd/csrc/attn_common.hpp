// Shared device helpers for the gfx950 (CDNA4) attention kernels: 64-lane wavefronts,
// v_mfma_f32_32x32x16_bf16 fragments, bf16 packing.  Compiled for gfx950 only.
#pragma once
#include <type_traits>
#include <utility>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "causal_order.hpp"
#include "xcd_order.hpp"

namespace fattn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// ---------------------------------------------------------------------------------------------
// v_mfma_f32_32x32x16_bf16:  D[32x32] += A[32x16] * B[16x32]
//   lane l, half h = l/32, n = l%32
//   A operand: 8 bf16 = A[n][8h .. 8h+7]        (row n, eight consecutive k)
//   B operand: 8 bf16 = B[8h .. 8h+7][n]        (column n, eight consecutive k)
//   C/D      : 16 f32, register r holds D[8*(r/4) + 4h + (r%4)][n]
// Because the k positions of A and B only have to agree with each other, any fixed permutation of
// the contraction index may be applied to both operands.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The same MFMA with the accumulator pinned to the architectural VGPRs, for kernels that also keep
// long-lived accumulators in the accumulation registers: the compiler picks one MFMA form per function,
// and with the accumulation form every value the vector ALU wants to read costs a v_accvgpr_read.
// Emitted by hand, so the compiler's hazard bookkeeping does not see it.  The caller must keep at
// least two other MFMAs between the last of these writing an accumulator and the first vector-ALU
// instruction that touches it (the result of an 8-pass MFMA is visible 11 issue cycles after issue).
// The B operand is held in the accumulation registers: operands that live for a whole kernel (a
// workgroup's own K / V fragments) then cost no architectural VGPRs.
// GUARD: two wait states in front, for kernel variants in which the register allocator moves an operand (part of an
// accumulator it has split, a fragment) into place right before the statement: an MFMA may read a register the vector
// ALU wrote two wait states later at the earliest, and the compiler keeps that distance only for its own MFMAs.
template <bool GUARD = false>
__device__ __forceinline__ void mfma32_vgpr_first_bacc(f32x16& acc, bf16x8 a, bf16x8 b) {
    if constexpr (GUARD) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "a"(b));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "a"(b));
}
template <bool GUARD = false>
__device__ __forceinline__ void mfma32_vgpr_bacc(f32x16& acc, bf16x8 a, bf16x8 b) {
    if constexpr (GUARD) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "a"(b));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "a"(b));
}
// Both operands in architectural registers (a kernel whose B fragments are too many for the accumulation file's
// free part).  After the last MFMA of a chain, mfma32_vgpr_settle spends the 11 wait states before its result may be
// read, for kernels that have no other MFMAs to put there.
// The two wait states in front: an operand the register allocator moved into place just before the statement was
// written by the vector ALU, and an MFMA may read such a register two wait states later at the earliest (the compiler
// keeps that distance for its own MFMAs, not for these).
__device__ __forceinline__ void mfma32_vgpr(f32x16& acc, bf16x8 a, bf16x8 b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma32_vgpr_settle(f32x16& acc) {
    asm volatile("s_nop 11" : "+v"(acc));
}
// ---------------------------------------------------------------------------------------------
// Fixed accumulation registers.  Inline assembly can only name a physical register by a literal, so the two
// register maps are written out once, here, and every statement below is generated from them; each row is checked
// against the rule it follows at compile time, so a wrong number does not build.
//   B slots:    slot s holds a 16-byte MFMA operand in a[128 + 4 s : 131 + 4 s]
//   acc tuples: tuple t holds a 32x32 fp32 accumulator block in a[16 t : 16 t + 15]
// ---------------------------------------------------------------------------------------------
#define FATTN_B_SLOTS(X) \
    X(0, 128, 129, 130, 131) \
    X(1, 132, 133, 134, 135) \
    X(2, 136, 137, 138, 139) \
    X(3, 140, 141, 142, 143) \
    X(4, 144, 145, 146, 147) \
    X(5, 148, 149, 150, 151) \
    X(6, 152, 153, 154, 155) \
    X(7, 156, 157, 158, 159) \
    X(8, 160, 161, 162, 163) \
    X(9, 164, 165, 166, 167) \
    X(10, 168, 169, 170, 171) \
    X(11, 172, 173, 174, 175) \
    X(12, 176, 177, 178, 179) \
    X(13, 180, 181, 182, 183) \
    X(14, 184, 185, 186, 187) \
    X(15, 188, 189, 190, 191) \
    X(16, 192, 193, 194, 195) \
    X(17, 196, 197, 198, 199) \
    X(18, 200, 201, 202, 203) \
    X(19, 204, 205, 206, 207) \
    X(20, 208, 209, 210, 211) \
    X(21, 212, 213, 214, 215) \
    X(22, 216, 217, 218, 219) \
    X(23, 220, 221, 222, 223) \
    X(24, 224, 225, 226, 227) \
    X(25, 228, 229, 230, 231) \
    X(26, 232, 233, 234, 235) \
    X(27, 236, 237, 238, 239) \
    X(28, 240, 241, 242, 243) \
    X(29, 244, 245, 246, 247) \
    X(30, 248, 249, 250, 251) \
    X(31, 252, 253, 254, 255)
#define FATTN_ACC_TUPLES(X) \
    X(0, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15) \
    X(1, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31) \
    X(2, 32, 33, 34, 35, 36, 37, 38, 39, 40, 41, 42, 43, 44, 45, 46, 47) \
    X(3, 48, 49, 50, 51, 52, 53, 54, 55, 56, 57, 58, 59, 60, 61, 62, 63) \
    X(4, 64, 65, 66, 67, 68, 69, 70, 71, 72, 73, 74, 75, 76, 77, 78, 79) \
    X(5, 80, 81, 82, 83, 84, 85, 86, 87, 88, 89, 90, 91, 92, 93, 94, 95) \
    X(6, 96, 97, 98, 99, 100, 101, 102, 103, 104, 105, 106, 107, 108, 109, 110, 111) \
    X(7, 112, 113, 114, 115, 116, 117, 118, 119, 120, 121, 122, 123, 124, 125, 126, 127)
#define FATTN_STR_(x) #x
#define FATTN_STR(x) FATTN_STR_(x)
#define FATTN_AREG(r) "a" FATTN_STR(r)
#define FATTN_ARANGE(lo, hi) "{a[" FATTN_STR(lo) ":" FATTN_STR(hi) "]}"
#define FATTN_CHECK_B_SLOT(I, R0, R1, R2, R3) \
    static_assert(R0 == 128 + 4 * I && R1 == R0 + 1 && R2 == R0 + 2 && R3 == R0 + 3, "row of FATTN_B_SLOTS")
#define FATTN_CHECK_ACC_TUPLE(I, R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15)                          \
    static_assert(R0 == 16 * I && R1 == R0 + 1 && R2 == R0 + 2 && R3 == R0 + 3 && R4 == R0 + 4 && R5 == R0 + 5 && R6 == R0 + 6 && \
                  R7 == R0 + 7 && R8 == R0 + 8 && R9 == R0 + 9 && R10 == R0 + 10 && R11 == R0 + 11 && R12 == R0 + 12 &&           \
                  R13 == R0 + 13 && R14 == R0 + 14 && R15 == R0 + 15, "row of FATTN_ACC_TUPLES")

// The same with the B operand pinned to accumulation registers a[128 + 4 SLOT : 131 + 4 SLOT], for a
// kernel whose 32 resident B fragments must stay put there (left to itself the register allocator
// homes some of them in architectural registers and copies them over before every use).
// MODE 0: acc = a b; 1: acc += a b; 2: acc = c + a b.
template <int SLOT, int MODE>
__device__ __forceinline__ void mfma32_vgpr_bpinned(f32x16& acc, bf16x8 a, bf16x8 b, const f32x16& c) {
    static_assert(SLOT >= 0 && SLOT < 32, "32 pinned fragments");
#define FATTN_PIN(I, R0, R1, R2, R3)                                                                                                        \
    FATTN_CHECK_B_SLOT(I, R0, R1, R2, R3);                                                                                                  \
    if constexpr (SLOT == I) {                                                                                                              \
        if constexpr (MODE == 0) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b));     \
        if constexpr (MODE == 1) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b));     \
        if constexpr (MODE == 2) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b), "v"(c)); \
    }
    FATTN_B_SLOTS(FATTN_PIN)
#undef FATTN_PIN
}

// The int8 counterpart (v_mfma_i32_32x32x32_i8: D[32x32] += A[32x32] * B[32x32], 16 consecutive int8 of the
// contraction per lane and operand, int32 accumulators in architectural VGPRs), same pinned B slots; the B
// value is the 128-bit carrier that pin_b_fragment returned.
template <int SLOT, int MODE>
__device__ __forceinline__ void mfma32i8_vgpr_bpinned(i32x16& acc, u32x4 a, bf16x8 b, const i32x16& c) {
    static_assert(SLOT >= 0 && SLOT < 32, "32 pinned fragments");
#define FATTN_PIN(I, R0, R1, R2, R3)                                                                                                      \
    if constexpr (SLOT == I) {                                                                                                            \
        if constexpr (MODE == 0) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b));     \
        if constexpr (MODE == 1) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b));     \
        if constexpr (MODE == 2) asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), FATTN_ARANGE(R0, R3)(b), "v"(c)); \
    }
    FATTN_B_SLOTS(FATTN_PIN)
#undef FATTN_PIN
}

// Moves a fragment into its pinned accumulation registers (the value the MFMAs above are given).
template <int SLOT>
__device__ __forceinline__ bf16x8 pin_b_fragment(u32x4 w) {
    bf16x8 out;
#define FATTN_PIN(I, R0, R1, R2, R3)                                                                                       \
    if constexpr (SLOT == I)                                                                                               \
        asm volatile("v_accvgpr_write_b32 " FATTN_AREG(R0) ", %1\n\tv_accvgpr_write_b32 " FATTN_AREG(R1) ", %2\n\t"        \
                     "v_accvgpr_write_b32 " FATTN_AREG(R2) ", %3\n\tv_accvgpr_write_b32 " FATTN_AREG(R3) ", %4"             \
                     : "=" FATTN_ARANGE(R0, R3)(out) : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
    FATTN_B_SLOTS(FATTN_PIN)
#undef FATTN_PIN
    return out;
}

// acc *= alpha for an accumulator tuple pinned to a[16 IDX : 16 IDX + 15], one register at a time through a
// single architectural register: rescaling accumulators that live in the accumulation registers
// through compiler-generated copies needs dozens of temporaries and ended in scratch spills.
template <int IDX>
__device__ __forceinline__ void rescale_pinned(f32x16& acc, float alpha) {
    static_assert(IDX >= 0 && IDX < 8, "eight pinned accumulator tuples");
    float tmp;
    // one register: read, multiply, one wait state, write back
#define FATTN_RS(r) "v_accvgpr_read_b32 %1, " FATTN_AREG(r) "\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\tv_accvgpr_write_b32 " FATTN_AREG(r) ", %1"
#define FATTN_PIN(I, R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15)                                      \
    FATTN_CHECK_ACC_TUPLE(I, R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15);                             \
    if constexpr (IDX == I)                                                                                                     \
        asm volatile(FATTN_RS(R0) "\n\t" FATTN_RS(R1) "\n\t" FATTN_RS(R2) "\n\t" FATTN_RS(R3) "\n\t" FATTN_RS(R4) "\n\t"        \
                     FATTN_RS(R5) "\n\t" FATTN_RS(R6) "\n\t" FATTN_RS(R7) "\n\t" FATTN_RS(R8) "\n\t" FATTN_RS(R9) "\n\t"        \
                     FATTN_RS(R10) "\n\t" FATTN_RS(R11) "\n\t" FATTN_RS(R12) "\n\t" FATTN_RS(R13) "\n\t" FATTN_RS(R14) "\n\t"   \
                     FATTN_RS(R15)                                                                                              \
                     : "+" FATTN_ARANGE(R0, R15)(acc), "=&v"(tmp) : "v"(alpha));
    FATTN_ACC_TUPLES(FATTN_PIN)
#undef FATTN_PIN
#undef FATTN_RS
}

// acc += a b with the accumulator pinned to a[16 IDX : 16 IDX + 15] (the tuples rescale_pinned works on) and both
// operands in architectural registers, emitted by hand: given the same fixed registers at every use, the accumulator
// never moves (left to the compiler's MFMA form, accumulators that a conditional rescale also touches travelled
// through architectural registers once per key tile).  Two wait states in front, as in mfma32_vgpr: the B operand may
// have been written, or moved into place, by the vector ALU just before.  mfma32_apinned_settle<IDX, WAIT> is the fence before the
// accumulators are read after the last tile: the one with WAIT spends the 11 wait states, and since volatile
// statements keep their order, fencing every accumulator after it orders all their reads behind that wait.
template <int IDX>
__device__ __forceinline__ void mfma32_apinned(f32x16& acc, bf16x8 a, bf16x8 b) {
    static_assert(IDX >= 0 && IDX < 8, "eight pinned accumulator tuples");
#define FATTN_PIN(I, R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15)                          \
    if constexpr (IDX == I) {                                                                                       \
        asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+" FATTN_ARANGE(R0, R15)(acc) : "v"(a), "v"(b)); \
    }
    FATTN_ACC_TUPLES(FATTN_PIN)
#undef FATTN_PIN
}
template <int IDX, bool WAIT>
__device__ __forceinline__ void mfma32_apinned_settle(f32x16& acc) {
    static_assert(IDX >= 0 && IDX < 8, "eight pinned accumulator tuples");
#define FATTN_PIN(I, R0, R1, R2, R3, R4, R5, R6, R7, R8, R9, R10, R11, R12, R13, R14, R15)     \
    if constexpr (IDX == I) {                                                                  \
        if constexpr (WAIT) asm volatile("s_nop 11" : "+" FATTN_ARANGE(R0, R15)(acc));         \
        else asm volatile("" : "+" FATTN_ARANGE(R0, R15)(acc));                                \
    }
    FATTN_ACC_TUPLES(FATTN_PIN)
#undef FATTN_PIN
}

// compile-time loop: f(std::integral_constant<int, 0>{}) ... f(std::integral_constant<int, N - 1>{})
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// row index inside a 32x32 accumulator block for register r of a lane in half h
__device__ __forceinline__ constexpr int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    f32x2 v = {lo, hi};
    bf16x2 b = __builtin_convertvector(v, bf16x2);   // v_cvt_pk_bf16_f32, round-to-nearest-even
    return __builtin_bit_cast(uint32_t, b);
}

// Waits until at most N of this wavefront's LDS reads are outstanding (they return in order); the vector
// memory and export counters are left alone.
template <int N>
__device__ __forceinline__ void wait_lds_reads() {
    static_assert(N >= 0 && N < 16, "lgkmcnt is a 4-bit field");
    __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}

__device__ __forceinline__ bf16x8 pack8(float a0, float a1, float a2, float a3, float a4, float a5, float a6,
                                        float a7) {
    u32x4 u = {pack_bf16(a0, a1), pack_bf16(a2, a3), pack_bf16(a4, a5), pack_bf16(a6, a7)};
    return __builtin_bit_cast(bf16x8, u);
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }   // v_exp_f32
__device__ __forceinline__ float log2_fast(float x) { return __builtin_amdgcn_logf(x); }    // v_log_f32

// exchange with the lane 32 positions away (the other half of the wave)
__device__ __forceinline__ float xhalf(float x) { return __shfl_xor(x, 32, 64); }

// max(x, xhalf(x)) without the way through the LDS crossbar: v_permlane32_swap_b32 makes the upper half of the first register
// change places with the lower half of the second.  By hand: given the same value twice, the compiler takes the two results of
// the builtin for one and folds the maximum away.  Two wait states in front, as it may read a register that the vector ALU has
// just written no earlier.
__device__ __forceinline__ float max_of_halves(float x) {
    float lo = x, hi = x;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
    return fmaxf(lo, hi);
}

// 16-byte global load of 8 bf16, zero when the predicate is false
__device__ __forceinline__ u32x4 ldg16(const uint16_t* p, bool ok) {
    u32x4 z = {0u, 0u, 0u, 0u};
    return ok ? *reinterpret_cast<const u32x4*>(p) : z;
}

typedef short s16x4 __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i receives element (i%4) of the four
// 8-byte rows addressed by lanes i/4, i/4+4, i/4+8, i/4+12 of the group.  When lane r of a group
// points at &X[k0 + r/4][c0 + 4*(r%4)] of a row-major tile X, lane i therefore receives
// X[k0+0..3][c0+i]: the group transposes a 4(k) x 16(column) block so that every lane ends up with
// four consecutive contraction elements of its own column.
__device__ __forceinline__ u32x2 lds_read_tr16(const uint16_t* p) {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
    return __builtin_bit_cast(u32x2, v);
}

// Elements between the rows of a tile in LDS.  The tiles of the kernels compiled for head dim 96 keep the layout of 128: six of
// eight steps of every contraction and three of four column blocks are computed, the last 32 columns of a row are never read.
template <int D>
constexpr int kRowPitch = D == 96 ? 128 : D;

// 16-byte-granule XOR swizzle of a row-major bf16 tile whose rows are kRowPitch<D> * 2 bytes (no padding).
// 16 consecutive rows get distinct bank groups for the same logical granule, and 4 consecutive rows
// land in 4 disjoint 64-byte bank groups: both access patterns used by the kernels (16-byte row
// reads, transposing 8-byte reads of a 4-row x 64-byte block) are conflict-free on the 64-bank LDS.
template <int D>
__device__ __forceinline__ constexpr int swz(int row) {
    return kRowPitch<D> == 128 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

// One wave-wide asynchronous copy global -> LDS: lane l delivers 16 (or 4) bytes to lds_dst + 16*l (4*l).
// The destination must be wave-uniform (it travels in M0).  Completion is tracked by vmcnt only, and
// the caller waits explicitly (wait_vm0 + barrier) before anyone reads the destination.
// The instruction is emitted by hand: when the compiler knows of a pending LDS-DMA it turns every
// following LDS-read wait into a full drain (lgkmcnt(0)), which defeats the read-ahead pipelines of
// the kernels.  Hidden from its wait-count bookkeeping, LDS reads of *other* buffers keep their exact
// counts.  Compiler-issued vmcnt waits stay correct: extra outstanding operations only make a
// counted wait stricter.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p);
}
// destination given as a wave-uniform LDS byte address
__device__ __forceinline__ void dma16(const void* gsrc, uint32_t lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(lds_byte_addr), "v"(gsrc) : "m0", "memory");
}
__device__ __forceinline__ void dma4(const void* gsrc, uint32_t lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" :: "s"(lds_byte_addr), "v"(gsrc) : "m0", "memory");
}
// ... and the source split into a wave-uniform base and a non-negative per-lane byte offset
__device__ __forceinline__ void dma16u(const void* gbase_wave_uniform, uint32_t lane_byte_off, uint32_t lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_byte_addr), "v"(lane_byte_off), "s"(gbase_wave_uniform) : "m0", "memory");
}
// The same copies in two halves, for software pipelines that place another instruction (an MFMA)
// between them instead of the s_nop: writing M0 and reading it in an LDS-DMA need one wait state.
// Nothing that writes M0 may come between the two halves.
__device__ __forceinline__ void dma_set_dst(uint32_t lds_byte_addr) {
    asm volatile("s_mov_b32 m0, %0" :: "s"(lds_byte_addr) : "m0");
}
__device__ __forceinline__ void dma16u_issue(const void* gbase_wave_uniform, uint32_t lane_byte_off) {
    asm volatile("global_load_lds_dwordx4 %0, %1" :: "v"(lane_byte_off), "s"(gbase_wave_uniform) : "memory");
}
__device__ __forceinline__ void dma4u_issue(const void* gbase_wave_uniform, uint32_t lane_byte_off) {
    asm volatile("global_load_lds_dword %0, %1" :: "v"(lane_byte_off), "s"(gbase_wave_uniform) : "memory");
}
// destination given as a pointer into LDS (wave-uniform)
__device__ __forceinline__ void dma16(const void* gsrc, void* lds_dst) { dma16(gsrc, lds_addr(lds_dst)); }
__device__ __forceinline__ void dma4(const void* gsrc, void* lds_dst) { dma4(gsrc, lds_addr(lds_dst)); }
__device__ __forceinline__ void dma16u(const void* gbase_wave_uniform, uint32_t lane_byte_off, void* lds_dst) {
    dma16u(gbase_wave_uniform, lane_byte_off, lds_addr(lds_dst));
}
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }   // vmcnt(0) only; a barrier follows
// At most N of this wavefront's vector memory operations are still outstanding (they complete in order).  The builtin is no
// access to memory for the compiler, which would move a plain load past it: the count would then stand for copies, and a read of
// their tile could come too early.  The empty statements keep every access on its side; the wait itself stays the builtin, so
// that the compiler knows what has landed.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
}

// Causal problems: the key walk of query unit qt grows with qt, and workgroups start in id order, so the longest
// walks must come first or they finish alone at the end.  Within the contiguous range of units that one XCD
// works through (whole heads where the counts allow), the order becomes: last unit of every head, then the
// units before them, and so on.  `wg`: unit id after xcd_remap, head-major, or, where eight does not divide the total, the
// workgroup's own (all of them in one order, dealt to the XCDs in turn); returns (qt, head) through refs.
template <bool SNAKE = false>
__device__ __forceinline__ void causal_longest_first(int wg, int n_qt, int total, int& qt, int& bh) {
    const int per_xcd = (total % 8 == 0) ? total / 8 : total;
    if (per_xcd % n_qt == 0) {
        const int heads = per_xcd / n_qt;
        const int base = wg / per_xcd * per_xcd, j = SNAKE && total % 8 == 0 ? snake_order(wg - base, per_xcd) : wg - base;
        qt = n_qt - 1 - j / heads;
        bh = base / n_qt + j % heads;
    } else {
        qt = n_qt - 1 - wg % n_qt;
        bh = wg / n_qt;
    }
}

struct Strides {
    int64_t b, h, n;   // element strides of a [B,H,N,D] bf16 view; the D stride is 1
};

// The 32 output rows of a wavefront, formed transposed (a lane owns row n and, per register group, four of its columns), to
// bf16 rows in memory.  Straight from the accumulators a store instruction touches 32 rows, 16 bytes of each, and the address
// unit takes four lanes of one cache line a clock: 64 clocks per instruction instead of 16, which every workgroup that has
// its compute unit to itself waits out at its end.  The rows pass through LDS instead (granules swizzled as in the tiles, so
// neither side has bank conflicts) and an instruction writes whole lines.  dK/dV of 256 key blocks, D = 128: 4.1 -> 1.9 us
// from the last step to the last store, D = 64 1.9 -> 1.1 us; forward and backward of B=3 H=16 128 x 138 D=128 31.4 -> 28.6 us,
// of B=4 H=16 1101 x 1101 D=128 with a key-padding mask 162 -> 155 us, of B=1 H=24 4608 x 4608 D=128 995 -> 985 us.
// own: 32 x kRowPitch<D> elements of LDS that only this wavefront touches; quad(db, g): columns 32 db + 8 g + 4 h .. + 3 of row n;
// rows: how many of the 32 exist; d: real head dim, a multiple of 8.  out and row_stride keep rows on 16 bytes.
template <int D, class F>
__device__ __forceinline__ void store_rows32(uint16_t* own, uint16_t* out, int64_t row_stride, int rows, int d, F&& quad) {
    constexpr int RS = kRowPitch<D>, GPR = RS / 8;
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x2*>(own + n * RS + (((4 * db + g) ^ swz<D>(n)) << 3) + 4 * h) = quad(db, g);
#pragma unroll
    for (int i = 0; i < GPR / 2; ++i) {
        const int row = (i * 64 + lane) / GPR, g = (i * 64 + lane) % GPR;
        const u32x4 w = *reinterpret_cast<const u32x4*>(own + row * RS + ((g ^ swz<D>(row)) << 3));
        if (row < rows && 8 * g < d) *reinterpret_cast<u32x4*>(out + row * row_stride + 8 * g) = w;
    }
}

// The same for fp32 partial sums: 32 x D floats of LDS; quad(db, g) as four floats.
template <int D, class F>
__device__ __forceinline__ void store_rows32_f32(float* own, float* out, int64_t row_stride, int rows, int d, F&& quad) {
    constexpr int GPR = D / 4;
    static_assert(GPR % 16 == 0, "the swizzle flips four bits of the granule");
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(own + n * D + (((8 * db + 2 * g + h) ^ (n & 15)) << 2)) = quad(db, g);
#pragma unroll
    for (int i = 0; i < GPR / 2; ++i) {
        const int row = (i * 64 + lane) / GPR, g = (i * 64 + lane) % GPR;
        const f32x4 w = *reinterpret_cast<const f32x4*>(own + row * D + ((g ^ (row & 15)) << 2));
        if (row < rows && 4 * g < d) *reinterpret_cast<f32x4*>(out + row * row_stride + 4 * g) = w;
    }
}

// The way in: 32 rows of a wavefront as MFMA fragments (lane: row n, 8 consecutive columns from 16 dc + 8 h on).  Loaded by the
// lanes that hold them, an instruction touches 32 rows, 32 bytes of each, at 64 clocks of the address unit; here four
// neighbouring lanes load 64 bytes of a row (16 clocks), and the rows pass through LDS, 32 columns at a time, two granules
// swizzled so that neither side has bank conflicts.  All loads first (load_rows32), then the way through LDS
// (fragments_of_rows32), so that several tensors can be in flight together.
// Rows at and past `rows` and columns at and past `d` (a multiple of 8) are zero.
template <int D>
__device__ __forceinline__ void load_rows32(u32x4 (&w)[D / 16], const uint16_t* base, int64_t row_stride, int rows, int d) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
        const int row = 16 * (i & 1) + (lane >> 2), col = 32 * (i >> 1) + 8 * (lane & 3);
        w[i] = ldg16(base + row * row_stride + col, row < rows && col < d);
    }
}
// own: 2 KiB of LDS that only this wavefront touches; take(dc, 16 bytes) for every dc < D / 16, given as a constant
template <int D, class F>
__device__ __forceinline__ void fragments_of_rows32(uint16_t* own, const u32x4 (&w)[D / 16], F&& take) {
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5, row = lane >> 2;
    uint16_t* const to = own + row * 32 + (((lane & 3) ^ ((row >> 2) & 3)) << 3);        // row + 16 has the same swizzle
    const uint16_t* const from = own + n * 32;
    static_for<D / 32>([&](auto c_tag) {
        constexpr int c = decltype(c_tag)::value;
        *reinterpret_cast<u32x4*>(to) = w[2 * c];
        *reinterpret_cast<u32x4*>(to + 16 * 32) = w[2 * c + 1];
        static_for<2>([&](auto u_tag) {
            constexpr int u = decltype(u_tag)::value;
            take(std::integral_constant<int, 2 * c + u>{}, *reinterpret_cast<const u32x4*>(from + (((2 * u + h) ^ ((n >> 2) & 3)) << 3)));
        });
    });
}

// Head dims below the compiled one (any multiple of 8, e.g. 80 on the 96-wide kernels) run zero-padded:
// fragments loaded straight from global memory are zero past the real head dim, tile copies re-read
// granule 0 of their row there (finite values that only ever meet those zero operands, or land in
// output rows past the real head dim, which are not stored), and stores skip those rows.
__device__ __forceinline__ int src_granule(int c, int d_real) { return c * 8 < d_real ? c : 0; }

// The 64 keep-mask bytes of one query row over a 64-key tile, as loaded by the kernels whose lanes own
// a query: keep(kb, r) is the byte of key 32*kb + acc_row(r, h).
struct MaskRow64 {
    u32x4 w[4];
    __device__ __forceinline__ void load(const uint8_t* row_tile) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const u32x4*>(row_tile + 16 * j);
    }
    // Clears the bytes of the keys at or past `limit` (relative to the first key of the tile): key-length and
    // causal exclusions then need no test of their own per element.  Meant for the few tiles they cut.
    __device__ __forceinline__ void restrict_to(int limit) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int c = min(max(limit - 4 * i, 0), 4);                  // bytes of dword i that stay
            const uint32_t m = c >= 4 ? 0xffffffffu : ((1u << (8 * c)) - 1u);
            w[i >> 2][i & 3] &= m;
        }
    }
    __device__ __forceinline__ bool keep(int kb, int r, int h) const {      // kb, r compile-time; h per lane
        const int d0 = 8 * kb + 2 * (r >> 2);                               // dword of the even half
        const uint32_t lo = w[d0 >> 2][d0 & 3], hi = w[(d0 + 1) >> 2][(d0 + 1) & 3];
        const uint32_t word = h ? hi : lo;
        return (word & (0xffu << (8 * (r & 3)))) != 0;
    }
};

enum MaskMode : int {
    kMaskU8 = 0,             // uint8, non-zero attends
    kMaskBf16Keep = 1,       // bf16, a value below 0.5 excludes (the public keep-mask convention of the reference)
    kMaskBf16Drop = 2,       // bf16, a value above 0.5 excludes (the convention of the reference's streaming entry point)
};

// flags of a 64 x 64 tile of (query, key), see mask_bits.hpp
constexpr uint8_t kTileAny = 1, kTileAllKeys = 2, kTileAllRows = 4;

struct MaskArgs {
    const int32_t* kv_len;   // [B] or null
    const uint8_t* mask;     // explicit mask or null; element type and meaning per mask_mode
    int64_t sb, sh, sq, sk;  // element strides over (b,h,q,k); 0 broadcasts
    int causal;              // key j > query i is excluded
    int rows16 = 0;          // uint8 keep-mask rows are contiguous along keys and 16-byte aligned (vector loads allowed)
    int mask_mode = kMaskU8;
    // the mask as bits (kernels instantiated for them only): words and flags of the planes, see mask_bits.hpp
    const uint64_t* bit_rows = nullptr;   // [plane][key tile][64 n_qt queries]
    const uint64_t* bit_cols = nullptr;   // [plane][query tile][64 n_kt keys]
    const uint8_t* tile_flags = nullptr;  // [plane][query tile][key tile]
    int bit_nqt = 0, bit_nkt = 0;         // tiles, padded to even numbers
    int plane_b = 0, plane_h = 0;         // plane of (b, h): b * plane_b + h * plane_h
    // additive bias on the scaled logits (forward only), fp32 or bf16, or null
    const void* bias = nullptr;
    int64_t bb = 0, bh = 0, bq = 0, bk = 0;   // element strides over (b,h,q,k); 0 broadcasts
    int bias_f32 = 1;
    float inv_scale = 1.f;   // 1 / softmax scale: the bias is folded into the raw scores as bias / scale
    // dropout of the probabilities (kernels instantiated with DROPOUT only): see drop_factor
    uint32_t drop_seed = 0;  // low 32 bits of the seed
    uint32_t drop_thr = 0;   // ceil(p * 2^24): an element is kept when its 24-bit uniform is >= this
    uint32_t drop_thr32 = 0; // drop_thr << 8, for the comparison with the whole 32-bit word
    float drop_scale = 1.f;  // 1 / (1 - p)
    uint32_t drop_cq = 0, drop_ck = 0;   // tiles of a chunked draw along queries and keys; drop_cq = 0: one draw over the tensor
};

// Factor that dropout applies to the probability of flat element index idx of the [B*H, Sq, Sk] probability tensor
// (low 32 bits): 0 or 1 / (1 - p).  The uniform is the reference's (src/rng/mod.rs:14-24, drawn over the whole
// tensor by src/autograd_v4/ops/sdpa.rs:229-231, :604-649): u = (xorshift32(seed ^ idx) >> 8) / 2^24, kept when
// u >= p, which in integers is (xorshift32(seed ^ idx) >> 8) >= ceil(p * 2^24).
__device__ __forceinline__ constexpr uint32_t xorshift32(uint32_t s) {
    s ^= s << 13;
    s ^= s >> 17;
    s ^= s << 5;
    return s;
}
__device__ __forceinline__ float drop_factor(const MaskArgs& m, uint32_t idx) {
    return (xorshift32(m.drop_seed ^ idx) >> 8) >= m.drop_thr ? m.drop_scale : 0.f;
}

// How a kernel draws.  xorshift32 is linear over GF(2): xorshift32(a ^ b) = xorshift32(a) ^ xorshift32(b).  Where the rows
// of the probability tensor start on multiples of 64 elements (Sk % 64 == 0) the index of an element is the index of the
// first element of its tile row XOR its offset, so one generator evaluation serves a row of a tile and every element costs
// an XOR with a constant, a comparison and a select; the factor 1 / (1 - p) is left to the sums.  (One evaluation per
// element, about ten vector instructions, more than doubles the vector work of the forward.)
enum DropMode : int {
    kDropNone = 0,
    kDropTiled = 1,      // any draw, chunked ones among them (drop_factor_at)
    kDropFlat = 2,       // one draw over the tensor
    kDropRows64 = 3,     // ... whose rows start on multiples of 64 elements
};

// The same for element (bh, qi, key) when the reference's operator is chunked (src/autograd_v4/ops/sdpa.rs:180-199,
// :444): it draws per tile of drop_cq x drop_ck (the last ones shorter) over the tile's own [B*H, q_t, k_t] tensor,
// under the seed derive_tile_seed gives (:600-602), whose low word is seed + k_offset (the query offset is shifted
// out of it).  drop_cq = 0 is the draw over the whole tensor.
__device__ __forceinline__ float drop_factor_at(const MaskArgs& m, uint32_t bh, uint32_t qi, uint32_t key, uint32_t Sq, uint32_t Sk) {
    if (m.drop_cq == 0) return drop_factor(m, (bh * Sq + qi) * Sk + key);
    const uint32_t qo = qi / m.drop_cq * m.drop_cq, ko = key / m.drop_ck * m.drop_ck;
    const uint32_t qt = min(m.drop_cq, Sq - qo), kt = min(m.drop_ck, Sk - ko);
    return (xorshift32((m.drop_seed + ko) ^ ((bh * qt + (qi - qo)) * kt + (key - ko))) >> 8) >= m.drop_thr ? m.drop_scale : 0.f;
}

// one element of an explicit mask, addressed in elements from the (batch, head) base: does it attend?
__device__ __forceinline__ bool mask_attends(const MaskArgs& m, const uint8_t* base, int64_t elem) {
    if (m.mask_mode == kMaskU8) return base[elem] != 0;
    const float v = __builtin_bit_cast(float, (uint32_t)reinterpret_cast<const uint16_t*>(base)[elem] << 16);
    return m.mask_mode == kMaskBf16Keep ? !(v < 0.5f) : !(v > 0.5f);
}
// (batch, head) base of an explicit mask
__device__ __forceinline__ const uint8_t* mask_head_base(const MaskArgs& m, int b, int hh) {
    return m.mask + (b * m.sb + hh * m.sh) * (m.mask_mode == kMaskU8 ? 1 : 2);
}

// What a kernel whose lanes own queries excludes besides keys past the key length and, with the causal flag, past the query.
enum Excl : int {
    kExNone = 0,
    kExRows16 = 1,       // uint8 keep-mask, rows contiguous and 16-byte aligned, Sk a multiple of the tile, no bias
    kExGeneral = 2,      // any keep-mask and / or bias, one element at a time
    kExBiasF32 = 3,      // (forward) an additive fp32 bias, contiguous along the keys, and no keep-mask, causal flag or key lengths
    kExBiasBf16 = 4,     // (forward) the same in bf16
    kExKeys = 5,         // a keep-mask that is the same for every query (a padded batch), no causal flag
    kExBits = 6,         // a keep-mask as bits, with the key lengths and the causal flag folded in
};

// The 64-key tiles that a keep-mask of keys leaves anything of, in LDS: the tiles attended whole first, then the others
// (the order of the tiles is irrelevant to the sums), and the 64 keep bits of every tile.  A padded batch walks the
// attended part of its sequences only, and nearly all of that without a test per element.
struct KeyTiles {
    static constexpr int kMaxTiles = 1024;            // 65536 keys: 10 KiB
    static __host__ __device__ int lds_bytes(int n_all) { return (n_all * 10 + 8 + 15) / 16 * 16; }
    uint64_t* bits;      // [n_all]
    uint32_t* counts;    // whole tiles, cut tiles
    uint16_t* list;      // [n_all]: whole tiles from the front, cut ones from the back
    int n_all, n_whole, n_tiles;

    // keep(key): does this key attend (false past the end)?  Every thread of the workgroup calls this; ends with a barrier.
    template <class F>
    __device__ __forceinline__ void build(void* lds, int n_keys, int nw, F&& keep) {
        n_all = (n_keys + 63) / 64;
        bits = static_cast<uint64_t*>(lds);
        counts = reinterpret_cast<uint32_t*>(bits + n_all);
        list = reinterpret_cast<uint16_t*>(counts + 2);
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll 4
        for (int t = wave; t < n_all; t += nw) {
            const uint64_t b = __ballot(keep(t * 64 + lane));
            if (lane == 0) bits[t] = b;
        }
        __syncthreads();
        sort_out([&](int t) { return bits[t] == ~0ull ? 2 : bits[t] != 0ull ? 1 : 0; });
    }
    // The same from what is known of the tiles: attended(t) says whether nothing (0), something (1) or all (2) of tile t is.
    template <class F>
    __device__ __forceinline__ void build_of_tiles(void* lds, int n_tiles_all, F&& attended) {
        n_all = n_tiles_all;
        bits = static_cast<uint64_t*>(lds);           // unused
        counts = reinterpret_cast<uint32_t*>(bits);
        list = reinterpret_cast<uint16_t*>(counts + 2);
        sort_out(attended);
    }
    template <class F>
    __device__ __forceinline__ void sort_out(F&& attended) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (wave == 0) {
            int whole = 0, cut = 0;
            for (int t0 = 0; t0 < n_all; t0 += 64) {
                const int a = t0 + lane < n_all ? attended(t0 + lane) : 0;
                const bool is_whole = a == 2, is_cut = a == 1;
                const uint64_t mw = __ballot(is_whole), mc = __ballot(is_cut), below = (1ull << lane) - 1ull;
                if (is_whole) list[whole + __popcll(mw & below)] = (uint16_t)(t0 + lane);
                if (is_cut) list[n_all - 1 - (cut + __popcll(mc & below))] = (uint16_t)(t0 + lane);
                whole += __popcll(mw);
                cut += __popcll(mc);
            }
            if (lane == 0) {
                counts[0] = (uint32_t)whole;
                counts[1] = (uint32_t)cut;
            }
        }
        __syncthreads();
        n_whole = __builtin_amdgcn_readfirstlane(counts[0]);
        n_tiles = n_whole + __builtin_amdgcn_readfirstlane(counts[1]);
    }
    // the j-th tile of the walk
    __device__ __forceinline__ int tile(int j) const {
        return __builtin_amdgcn_readfirstlane(list[j < n_whole ? j : n_all - 1 - (j - n_whole)]);
    }
};

// Batches of unequal key lengths: workgroups start in id order, so the longest walks must come first or the last of them run
// alone at the end.  `bh` counts (batch, head) slices in start order; the result is the slice it stands for when the batches
// come in the order of descending weight (ties in their own order; the heads of a batch stay in theirs).  The weight of a
// batch is its key length, or, with a keep-mask of keys, how many of 64 keys spread over the sequence it attends: a guess that
// costs one load per batch and lane and decides nothing but the order.  Every lane of the workgroup calls this and every
// workgroup gets the same order.  More batches than `kMaxRanked` come as they are (a rank costs two instructions per batch,
// a sampled mask a load per batch).
// Lengths 30, 50, 80 and 100 % of Sk in ascending order: forward and backward of B=4 H=16 1024 x 2049 D=64 150 -> 134 us with
// key lengths, of 1101 x 1101 D=128 192 -> 181 us with a mask.
template <bool KEYS>
__device__ __forceinline__ int longest_batches_first(int bh, int B, int H, int Sk, const MaskArgs& m) {
    constexpr int kMaxRanked = KEYS ? 16 : 64;
    if (B < 2 || B > kMaxRanked) return bh;
    const int lane = threadIdx.x & 63;
    int w = -1;                                           // lane j: the weight of batch j
    if constexpr (KEYS) {
        const int key = (int)(((int64_t)(2 * lane + 1) * Sk) >> 7);
#pragma unroll 4
        for (int j = 0; j < B; ++j) {
            const int len = m.kv_len ? min(Sk, m.kv_len[j]) : Sk;
            const int kept = __popcll(__ballot(key < len && mask_attends(m, mask_head_base(m, j, 0), (int64_t)key * m.sk)));
            w = lane == j ? kept : w;
        }
    } else {
        if (lane < B) w = min(max(m.kv_len[lane], 0), Sk);
    }
    int rank = 0;                                         // of batch `lane`
    for (int j = 0; j < B; ++j) {
        const int wj = __builtin_amdgcn_readlane(w, j);
        rank += (wj > w || (wj == w && j < lane)) ? 1 : 0;
    }
    const int r = bh / H;
    const int b = __ffsll((unsigned long long)__ballot(lane < B && rank == r)) - 1;
    return __builtin_amdgcn_readfirstlane(b) * H + bh % H;
}

}  // namespace fattn
