// fp32 values as three bf16, for products on v_mfma_f32_16x16x32_bf16.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), all rounded to nearest even: both subtractions are exact, h
// takes eight of the 24 bits, m eight of the at most 16 that are left, and l the rest, so the sum is x itself (down to 2^-110; what
// lies below 2^-133 of a smaller x is rounded off). Of the nine products of two such numbers six are summed; the others
// (m l, l m, l l) are below 2^-26 of the whole product. A product of bf16 numbers is exact in fp32, and six of these instructions
// take 96 cycles for the 16 x 16 x 32 multiply-adds that take v_mfma_f32_16x16x4_f32 256: 298 TFLOP/s against 151 in a loop of
// nothing else (the device holds 1.75 GHz under the former, 2.4 GHz under the latter).
//
// The sums of 32 k start from zero and are added to the running sum with an fp32 addition: one rounding at the sum's size per 32 k
// where the fp32 instruction makes eight. Relative error against 64 bits (2-norm, normal operands) of 576 products 9.4e-8 (fp32
// instruction 4.3e-7; six products added straight to the running sum 3.6e-7), of 4096 products 2.2e-7 (1.15e-6).
//
// An infinity or NaN in an operand makes every sum it takes part in non-finite (inf * 0 for the parts that are zero), also where
// the fp32 sum would be an infinity: a kernel looks at its sums and repeats those of a tile with fp32 instructions if one
// of them is not finite.
#pragma once
#include "common.h"

namespace sofie {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));

struct Split8 {
   v8b h, m, l;
};

// Eight numbers as h, m and l, two at a time: v_cvt_pk_bf16_f32, the two bf16 as fp32 by a shift and a mask, subtractions: eleven
// instructions a pair (18 where the compiler converted each number by itself). x - h as a sum of products of bf16 (v_dot2c_f32_bf16, seven
// a pair) waits for the matrix pipe: ns for each v_mfma_f32_16x16x32_bf16, two wavefronts on a SIMD: 7.4 alone, 7.5 with two
// conversions or subtractions behind it, 9.1 with three; 14.6 with two dot products.
__device__ __forceinline__ void split8(const float (&x)[8], v4i (&d)[3])
{
   v4f r0, r1;
#pragma unroll
   for (int p = 0; p < 4; ++p) {
      r0[p] = x[2 * p];
      r1[p] = x[2 * p + 1];
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

// The same for operands that are laid out once and read back as fp32 (joined) where sums are repeated: an x that is not finite is h
// alone, and one that would round up to infinity has its last bits cut off in h instead.
__device__ __forceinline__ Split8 split8_exact(const float (&x)[8])
{
   Split8 s;
#pragma unroll
   for (int e = 0; e < 8; ++e) {
      const bool finite = (__float_as_uint(x[e]) & 0x7f800000u) != 0x7f800000u;
      s.h[e] = (__bf16)x[e];
      if (finite && (__float_as_uint((float)s.h[e]) & 0x7f800000u) == 0x7f800000u)
         s.h[e] = (__bf16)__uint_as_float(__float_as_uint(x[e]) & 0xffff0000u);
      const float r = finite ? x[e] - (float)s.h[e] : 0.0f;
      s.m[e] = (__bf16)r;
      s.l[e] = (__bf16)(r - (float)s.m[e]);
   }
   return s;
}

__device__ __forceinline__ float joined(__bf16 h, __bf16 m, __bf16 l)
{
   return (float)h + ((float)m + (float)l);
}

}  // namespace sofie
