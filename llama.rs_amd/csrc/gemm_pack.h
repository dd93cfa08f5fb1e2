// Input layout of the prompt GEMM (gemm.hip), written by the kernels that
// produce its rows (prefill.hip) or by launch_gemm_pack.
//
// The rows come in tiles of 32 and the row length K in super-blocks of 256.
// The bytes of one (row tile, super-block) are contiguous and in the order in
// which the matrix cores read them, so that the GEMM copies them to LDS
// without an address computation per row and every operand read of a
// wavefront is one contiguous KB: K-step t (16 of them, 16 elements each)
// holds for lane m + 32 hf the eight elements
//   64 (t >> 2) + 32 ((t >> 1) & 1) + 16 hf + 8 (t & 1) + {0,2,1,3,4,6,5,7}
// of row m: the order in which the weights' nibbles unpack two at a time from
// 32-bit words (elements i and i + 2 of a word's four bytes sit 16 bits apart).
//   precision 3: per K-step 1 KB of f16 hi, then 1 KB of f16 lo (hi + lo = 22
//     bits of x * 2^-e, or 2^-25 in absolute terms where that is coarser; e the
//     super-block's own), after the 16 steps 1 KB of sub-block sums (lane m: the
//     f16 hi of the eight 32-element sums of row m, lane m + 32: their lo) for
//     the K-quant minima, then the 32 rows' 2^e in f32 (padded to 1 KB).
//     e is the least for which every element and every sub-block sum is below
//     2^15 times 2^e: an element keeps its 22 bits down to 2^-17 of the largest
//     of its super-block, 16 bits (a bf16 hi + lo pair's) down to 2^-21, and an
//     absolute 2^-40 of the largest below.  (With e fixed by 32 times the largest
//     element, which no sum can exceed, it was 2^-35: beside one element of 2^20
//     the error of N(0, 1) elements was 3.5e-5, now 1.1e-6; bf16 pairs have 2.5e-6.)
//   precision 1: per K-step 1 KB of bf16
#pragma once

#include "lrs_internal.h"

namespace lrs {

constexpr uint32_t GP_SUMS = 32768, GP_SCALE = 33792;  // offsets in a precision-3 block

// the f16 element pair order inside eight elements
__device__ __forceinline__ uint32_t gp_slot(uint32_t i) { return (i & 4) | ((i & 1) << 1) | ((i >> 1) & 1); }

// Eight consecutive elements v (element 8 c of row `row`) into the planes p of
// a GEMM input of row length K = 256 nsb.  Called by all 32 lanes of a half
// wavefront with consecutive c (one super-block of the row: c % 32 = lane % 32).
template <int PREC>
__device__ __forceinline__ void gp_store8(const float (&v)[8], uint32_t row, uint32_t c, uint32_t nsb,
                                          uint8_t *__restrict__ p) {
    const uint32_t c8 = c & 31;  // chunk in the super-block: group j, half of 32, hf, 8-element part
    const uint32_t t = 4 * (c8 >> 3) + 2 * ((c8 >> 2) & 1) + (c8 & 1), hf = (c8 >> 1) & 1;
    uint8_t *const b = p + ((size_t)(row >> 5) * nsb + (c >> 5)) * gemm_block_bytes(PREC);
    const uint32_t lane16 = 16 * ((row & 31) + 32 * hf);
    if constexpr (PREC == 1) {
        typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_p;
        bf16x8_p h;
#pragma unroll
        for (int i = 0; i < 8; i++) h[gp_slot(i)] = (__bf16)v[i];
        *reinterpret_cast<bf16x8_p *>(b + 1024 * t + lane16) = h;
    } else {
        typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_p;
        // The largest |x| / 32 and sub-block sum of x / 32, which it bounds.  A
        // sub-block is four lanes: the first two steps of the one reduction run
        // beside the other's, so that five shuffles follow one another, not seven
        // (a pack of 64 rows of 5120 5.0 us with them after one another, 4.8).
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
        float w[8];  // no sum of these overflows
#pragma unroll
        for (int i = 0; i < 8; i++) w[i] = v[i] * 0.03125f;
        float s = ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
#pragma unroll
        for (int o = 1; o <= 2; o *= 2) {
            mx = fmaxf(mx, __shfl_xor(mx, o, 64));
            s += __shfl_xor(s, o, 64);
        }
        mx = fmaxf(mx * 0.03125f, fabsf(s));
#pragma unroll
        for (int o = 4; o <= 16; o *= 2) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        int ex;
        (void)frexpf(mx, &ex);  // mx < 2^ex: elements and sums below 2^(ex + 5)
        ex = mx > 0.f ? (ex < -100 ? -100 : ex) : 0;
        f16x8_p h, l;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float x = ldexpf(v[i], 10 - ex);
            const _Float16 xh = (_Float16)x;
            h[gp_slot(i)] = xh;
            l[gp_slot(i)] = (_Float16)(x - (float)xh);
        }
        *reinterpret_cast<f16x8_p *>(b + 2048 * t + lane16) = h;
        *reinterpret_cast<f16x8_p *>(b + 2048 * t + 1024 + lane16) = l;
        if ((c8 & 3) == 0) {
            s = ldexpf(s, 15 - ex);
            const _Float16 sh = (_Float16)s;
            _Float16 *sp = reinterpret_cast<_Float16 *>(b + GP_SUMS + 16 * (row & 31)) + gp_slot(c8 >> 2);
            sp[0] = sh;
            sp[256] = (_Float16)(s - (float)sh);
        }
        if (c8 == 0) *reinterpret_cast<float *>(b + GP_SCALE + 4 * (row & 31)) = ldexpf(1.0f, ex - 10);
    }
}

}  // namespace lrs
