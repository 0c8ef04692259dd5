// fp32 values as three bf16, for products on v_mfma_f32_16x16x32_bf16.
//
// 2^16 x = h + m + l with h = bf16(2^16 x), m = bf16(2^16 x - h), l = bf16(2^16 x - h - m), all rounded to nearest even: both subtractions
// are exact, h takes eight of the 24 bits, m eight of the at most 16 that are left, and l the rest, so the sum is 2^16 x itself. The
// factor puts the last bit of the smallest fp32 number, 2^-149, on the last bit of the smallest bf16, 2^-133 (without it numbers below
// 2^-110 lost bits: relative error 5.6e-7 at 2^-114, 2.3e-3 at 2^-126); sums are 2^32 times too large and are multiplied by
// 2^-32 behind the loop (UNSCALE). The factor costs a multiplication per number split: 1500 x 1001 x 1111 28.4 -> 29.2 us, 4096^3 792 -> 820,
// 256x64x56x56 -> 128, 3x3 597 -> 605, transposed 64x128x28x28 -> 64, 4x4 s2 90.3 -> 93.3; 66 random convolutions 0.8 % in the median.
//
// Of the nine products of two such numbers six are summed; the others (m l, l m, l l) are together at most 2^-24 of the whole product
// (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|; 1 + 2^-8 - 2^-17 by itself), and 2^-27 of it in the root mean square over random operands. A product
// of bf16 numbers is exact in fp32, and six of these instructions take 96 cycles for the 16 x 16 x 32 multiply-adds that take
// v_mfma_f32_16x16x4_f32 256: 298 TFLOP/s against 151 in a loop of nothing else (the device holds 1.75 GHz under the former, 2.4 GHz
// under the latter).
//
// The sums of 32 k start from zero and are added to the running sum with an fp32 addition: one rounding at the sum's size per 32 k
// where the fp32 instruction makes eight. Relative error against 64 bits (2-norm, normal operands) of 576 products 9.4e-8 (fp32
// instruction 4.3e-7; six products added straight to the running sum 3.6e-7), of 4096 products 2.2e-7 (1.15e-6).
//
// An infinity or NaN in an operand makes every sum it takes part in non-finite (inf * 0 for the parts that are zero), also where
// the fp32 sum would be an infinity, and so do finite operands from 2^111 and sums from 2^95 on: a kernel looks at its sums and repeats
// those of a tile with fp32 instructions on the operands as they were given if one of them is not finite.
#pragma once
#include "common.h"

namespace sofie {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));

// Eight numbers as h, m and l, two at a time: v_cvt_pk_bf16_f32, the two bf16 as fp32 by a shift and a mask, subtractions: eleven
// instructions a pair behind the two multiplications (18 where the compiler converted each number by itself). x - h as a sum of products of bf16 (v_dot2c_f32_bf16, seven
// a pair) waits for the matrix pipe: ns for each v_mfma_f32_16x16x32_bf16, two wavefronts on a SIMD: 7.4 alone, 7.5 with two
// conversions or subtractions behind it, 9.1 with three; 14.6 with two dot products.
__device__ __forceinline__ void split8(const float (&x)[8], v4i (&d)[3])
{
   v4f r0, r1;
#pragma unroll
   for (int p = 0; p < 4; ++p) {
      r0[p] = __fmul_rn(x[2 * p], 65536.0f);
      r1[p] = __fmul_rn(x[2 * p + 1], 65536.0f);
   }
#pragma unroll
   for (int part = 0; part < 3; ++part) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
         const unsigned both = f32x2_to_bf16x2(r0[p], r1[p]);
         d[part][p] = (int)both;
         if (part < 2) {
            r0[p] -= __uint_as_float(both << 16);
            r1[p] -= __uint_as_float(both & 0xffff0000u);
         }
      }
   }
}

// What a sum of such products is multiplied by.
constexpr float UNSCALE = 0x1p-32f;

}  // namespace sofie
