// Main loops on 16x16 MFMAs: the instruction, where its operands lie in LDS, and the way back to the layout of 32x32 ones, which the epilogues know.
//
// At the board's power limit, where the long loops run, products per second are products per joule.  A 16x16 MFMA takes as many cycles per
// product as a 32x32 one and less energy: fragment reads and MFMAs alone, 64x128 per wave, eight waves per CU, sustain 1505 TFLOP/s on 32x32
// and 1676 on 16x16 ones (fp16, normal operands), 3083 and 3503 TOPS (uniform int8; profiles/probe_mfma_16x16_and_32x32.md).  In the order of snake16() a fragment
// of B meets four of A and the next one starts with the last of these, so one operand changes at a time: 1661 and 3473 without the turn.
// Whole launches on 256x256 tiles, 32x32 -> 16x16, calls behind each other: fp16 8192x27392x4096 as [n,k] 1533 -> 1409 us (1199 -> 1304 TFLOP/s),
// fp16 all-gather 4 x [610,13632] x [13632,2560] 355 -> 339, 8144x5120x1696 167.5 -> 159.9.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_fused_kernel.h"

namespace catcoc {

template <uint32_t DT> struct Acc16Of { using type = v4f; };
template <> struct Acc16Of<DT_I8> { using type = v4i; };

// 64 bytes of k of 16 rows of A (lane: row lane & 15, 16-byte piece lane >> 4) and of 16 columns of B the same way.  Element r of a lane's result:
// row 4 * (lane >> 4) + r, column lane & 15.
template <uint32_t DT>
__device__ __forceinline__ typename Acc16Of<DT>::type mfma16(v4i a, v4i b, typename Acc16Of<DT>::type c)
{
    if constexpr (DT == DT_I8) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
    } else if constexpr (DT == DT_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    }
}

constexpr int snake16(int j, int i, int rows) { return j & 1 ? rows - 1 - i : i; }

// B as [k,n], a stage of rows of k: the 16-byte column piece q of row `row` lies at slot q ^ b16_slot(row).  A half wave's transposing read takes 16
// columns of eight rows of 4-byte lanes (2-byte elements: rows 0-3 and 8-11 of a step) or of sixteen of 1-byte ones (0-7 and 16-23), and they lie in all banks once.
template <int ES>
__device__ __forceinline__ uint32_t b16_slot(uint32_t row)
{
    if constexpr (ES == 1) return ((row & 7u) << 1) | ((row >> 4) & 1u);
    else return ((row & 3u) << 2) | (((row >> 3) & 1u) << 1);
}

// Rows of 64 bytes of k: piece c of row `row` lies at slot c ^ k16_slot(row).  A 16-byte read is served 16 lanes at a time, of rows 0-3 and 12-15
// the one piece and of rows 4-11 the next, or the other way round.
__device__ __forceinline__ uint32_t k16_slot(uint32_t row)
{
    const uint32_t q = row >> 2;
    return (((q ^ (q >> 1)) & 1u) << 1) | ((q >> 1) & 1u);
}

// The same values, 32 columns to a register as with 32x32 MFMAs: block (2 * mb + br, 2 * nb + bc) of 16x16 holds rows 16 * br + 4 * (lane >> 4) + r; of
// a 32x32 block a lane then holds column lane & 31 and rows 16 * (reg >> 3) + 8 * (lane >> 5) + (reg & 7).  (Bit 4 of the lane, four rows, changes
// places with bc.  The rows of 32x32 MFMAs' registers would take as many swaps again.)
template <uint32_t DT, int MB, int NB>
__device__ __forceinline__ void acc16_to_32(const typename Acc16Of<DT>::type (&x)[2 * MB][2 * NB], typename AccOf<DT>::type (&acc)[MB][NB])
{
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int br = 0; br < 2; ++br)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto e0 = x[2 * mb + br][2 * nb][r], e1 = x[2 * mb + br][2 * nb + 1][r];
                    const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, e0), __builtin_bit_cast(uint32_t, e1), false, false);
                    const uint32_t s0 = s[0], s1 = s[1];
                    acc[mb][nb][8 * br + r] = __builtin_bit_cast(std::remove_const_t<decltype(e0)>, s0);
                    acc[mb][nb][8 * br + 4 + r] = __builtin_bit_cast(std::remove_const_t<decltype(e0)>, s1);
                }
}

}  // namespace catcoc
