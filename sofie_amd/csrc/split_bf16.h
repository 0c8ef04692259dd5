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

__device__ __forceinline__ Split8 split8(const float (&x)[8])
{
   Split8 s;
#pragma unroll
   for (int e = 0; e < 8; ++e) {
      s.h[e] = (__bf16)x[e];
      const float r = x[e] - (float)s.h[e];
      s.m[e] = (__bf16)r;
      s.l[e] = (__bf16)(r - (float)s.m[e]);
   }
   return s;
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

// Sums over 32 k: the small products first.
__device__ __forceinline__ v4f mma_split(const v8b (&a)[3], const v8b (&b)[3])
{
   v4f t = {0.0f, 0.0f, 0.0f, 0.0f};
   t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], t, 0, 0, 0);
   t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], t, 0, 0, 0);
   t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], t, 0, 0, 0);
   t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], t, 0, 0, 0);
   t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], t, 0, 0, 0);
   return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], t, 0, 0, 0);
}

__device__ __forceinline__ bool not_finite(v4f v)
{
   bool bad = false;
#pragma unroll
   for (int e = 0; e < 4; ++e) bad = bad || (__float_as_uint(v[e]) & 0x7f800000u) == 0x7f800000u;
   return bad;
}

}  // namespace sofie
