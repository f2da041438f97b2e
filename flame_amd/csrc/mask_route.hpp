// Which kernels serve a keep-mask that differs by query: those that walk by its bits (mask_bits.hpp) or those that read it.
#pragma once
#include <stdint.h>

namespace fattn {

// its rows are contiguous along the keys and on 16 bytes, all of them
inline bool mask_rows16(const void* mask, int64_t sb, int64_t sh, int64_t sq, int64_t sk) {
    return mask && sk == 1 && (reinterpret_cast<uintptr_t>(mask) | (uintptr_t)sb | (uintptr_t)sh | (uintptr_t)sq) % 16 == 0;
}

// The kernels that read the mask lose only where they cannot load it as vectors (4 to 5 times the time: bits from 36 tiles of
// 64 x 64 on, below which a step's two further launches weigh more) or where tiles can be left out, which the host does not know.  So
// where they can, bits are taken from the size on from which documents packed into a sequence gain and masks of chance, whose
// tiles are all cut, lose little.  Time by rows / time by bits, B x H = 1 x 16 to 8 x 16, D = 64 to 128, chance and four documents:
//   one mask for all heads      512 x 512   768          1024         1280         1536         2048
//     forward   chance          0.73-0.95   0.81-1.04    0.85-1.04    0.86-1.06    0.88-1.08    0.96-1.13
//               documents       0.81-0.96   0.83-1.27    0.92-1.32    0.97-1.58    1.14-1.50    1.07-1.31
//     backward  chance          0.86-1.01   0.93-1.07    0.94-1.04    0.96-1.10    0.97-1.10    0.99-1.14
//               documents       0.90-1.08   0.95-1.35    0.96-1.34    0.98-1.52    1.17-1.41    1.13-1.29
//   a mask for every head
//     forward   chance          0.69-0.84   0.76-0.87    0.71-0.84    0.82-0.93    0.80-0.93    0.78-0.89
//               documents       0.70-0.84   0.77-0.91    0.79-0.95    0.85-1.14    0.85-0.98    0.84-0.96
//     backward  chance          0.85-1.00   0.89-0.98    0.89-0.99    0.92-1.05    0.91-1.06    0.90-1.03
//               documents       0.89-1.01   0.92-1.05    0.97-1.15    1.05-1.29    1.07-1.08    1.05-1.12
// (each head's own mask is read once by the forward: the pass over it costs what the bits save).  With the causal flag on top,
// documents, forward: one mask 0.88-1.09, at 1024 1.08-1.45, from 1280 on 0.98-1.82; one for every head 0.60-1.10.
inline bool mask_bits_pay(bool backward, bool rows16, bool per_head, int64_t row_stride, int Sq, int Sk, bool causal) {
    const int64_t tiles = (int64_t)((Sq + 127) / 128 * 2) * ((Sk + 127) / 128 * 2);
    // (what the kernels of either direction ask of the call besides: dK/dV 32-bit offsets within 64 rows)
    const bool vectors = rows16 && (backward ? !causal && Sk % 128 == 0 && Sq % 64 == 0 && 64 * row_stride < (int64_t)1 << 31 : Sk % 64 == 0);
    if (!vectors) return tiles >= 36;
    return backward ? tiles >= 256 : !per_head && tiles >= (causal ? 256 : 400);
}

}  // namespace fattn
