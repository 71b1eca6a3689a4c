// Integers as signed bytes for the matrix cores: v_mfma_i32_16x16x64_i8 multiplies 16 rows by 16
// columns over 64 products of signed bytes, exactly in int32. A wider integer is its balanced
// base-256 digits, sum_i d_i 2^(8 i) with d_i in [-128, 127]: byte i of (x + 0x808080), its top bit
// flipped (digits 0 to 2; what is left above them is digit 3).
#pragma once

#include "insitu_internal.h"

namespace insitu {

typedef int v4i __attribute__((ext_vector_type(4)));

// Operands: lane = (row or column l % 16, 16 consecutive products of group l / 16), a byte each.
// Result: lane = (column l % 16, rows 4 (l / 16) ..).
__device__ __forceinline__ v4i mma(v4i rows, v4i cols, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(rows, cols, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);         // selector bytes 0-3: lo, 4-7: hi, 12: zero
}
// The balanced digits 0 to 2 of x as bytes 0 to 2, and digit 3 as byte 3 (x at most 2^31 - 1 - 0x808080:
// from there on x + 0x808080 leaves int32).
__device__ __forceinline__ uint32_t balanced(int32_t x) { return ((uint32_t)x + 0x808080u) ^ 0x808080u; }

// The digits of 16 key centroids, dg[i][j] holding digit i of centroids 4 j .. 4 j + 3.
// 16 codes of KB bits, LSB first in x, to their centroids' digits: o[i] the digit-i bytes of 16
// products, in the codes' order, or with 4-bit codes the even and the odd codes of each 8 in turn
// (the order the nibbles come in; channel_of).
template <int KB>
__device__ __forceinline__ void expand16(uint64_t x, const uint32_t (&dg)[3][4], v4i (&o)[3]) {
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    uint32_t sel[4];
    if constexpr (KB == 4) {
        sel[0] = lo & 0x0F0F0F0Fu;
        sel[1] = (lo >> 4) & 0x0F0F0F0Fu;
        sel[2] = hi & 0x0F0F0F0Fu;
        sel[3] = (hi >> 4) & 0x0F0F0F0Fu;
    } else if constexpr (KB == 3) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t y = (uint32_t)(x >> (12 * w)) & 0xFFFu, z = (y | y << 10) & 0x003F003Fu;
            sel[w] = (z | z << 5) & 0x07070707u;
        }
    } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t y = (lo >> (8 * w)) & 0xFFu, z = (y | y << 12) & 0x000F000Fu;
            sel[w] = (z | z << 6) & 0x03030303u;
        }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        if constexpr (KB == 4) {
            const uint32_t top = perm(0u, 0u, ((sel[w] >> 3) & 0x01010101u) + 0x0C0C0C0Cu);   // FF where code >= 8
            const uint32_t s7 = sel[w] & 0x07070707u;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const uint32_t a = perm(dg[i][1], dg[i][0], s7), c = perm(dg[i][3], dg[i][2], s7);
                o[i][w] = (int)((a & ~top) | (c & top));
            }
        } else {
#pragma unroll
            for (int i = 0; i < 3; ++i) o[i][w] = (int)perm(dg[i][1], dg[i][0], sel[w]);
        }
    }
}
// The channel, within 16, of product byte j (expand16's order).
__host__ __device__ constexpr int channel_of(int kb, int j) {
    return kb == 4 ? 8 * (j / 8) + 2 * (j % 4) + (j / 4) % 2 : j;
}

}  // namespace insitu
