// fp32 products: what their kernels share.
#pragma once
#include "common.h"

namespace sofie {

struct GemmF32Args {
   const float *A, *B, *bias;
   float *Y;
   int M, N, K, lda, ldb, ldy;
   int transA, transB;
   float alpha, beta;
   int bias_kind, relu;
   // stacked products (blockIdx.z + z0 = index of the product, row-major over the n_lead leading dimensions):
   // element strides of A and B along each leading dimension (0 where the operand is broadcast), Y is dense
   int n_lead, z0;
   int lead[SOFIE_GEMM_MAX_LEAD];
   long long sa[SOFIE_GEMM_MAX_LEAD], sb[SOFIE_GEMM_MAX_LEAD];
   long long stride_y;
   // k_gemm_f32_dma with K in slices (gridDim.y > 1): a slice's raw sums go to partial [slice][M][N]
   float *partial;
};

// Workgroup id -> tile, in groups of 4 rows of tiles, so that the workgroups in flight share rows of A and columns of B in an
// L2. Workgroups are dealt to the 8 XCDs in turn: renumbered so that an XCD (an L2) works on consecutive tiles.
__device__ __forceinline__ void tile_of(int pid, int tiles_m, int tiles_n, int &tm, int &tn)
{
   {
      const int tiles = tiles_m * tiles_n, xcd = pid & 7, base = tiles >> 3, rem = tiles & 7;
      pid = (pid >> 3) + xcd * base + (xcd < rem ? xcd : rem);
   }
   const int width = 4 * tiles_n, group = pid / width, first = group * 4;
   const int gsize = tiles_m - first < 4 ? tiles_m - first : 4;
   tm = first + (pid % width) % gsize;
   tn = (pid % width) / gsize;
}

// A, B and Y of product `index` of a stack (row-major over the leading dimensions, last dimension fastest).
__device__ __forceinline__ void select_product(GemmF32Args &g, long long index)
{
   long long rem = index, oa = 0, ob = 0;
   // (constant subscripts: with a run-time one the whole argument block would move to scratch memory)
#pragma unroll
   for (int d = SOFIE_GEMM_MAX_LEAD - 1; d >= 0; --d) {
      if (d >= g.n_lead) continue;
      const long long pos = rem % g.lead[d];
      rem /= g.lead[d];
      oa += pos * g.sa[d];
      ob += pos * g.sb[d];
   }
   g.A += oa;
   g.B += ob;
   g.Y += index * g.stride_y;
}

// The bias of columns n .. n + 3 where a row of it is given. (Requested ahead of a kernel's sums: four loads behind them for every
// four outputs were a third of the time of a product with a short K; 3274 x 7184 x 16 64 us, 2 of K on 3192 x 3280 36.)
__device__ __forceinline__ v4f bias_row4(const GemmF32Args &g, int n)
{
   v4f b = {0.0f, 0.0f, 0.0f, 0.0f};
   if (g.bias_kind == SOFIE_BIAS_ROW) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
         if (n + e < g.N) b[e] = g.bias[n + e];
   }
   return b;
}
// alpha * v + beta * bias, ReLU, for columns n .. n + 3 of row m; row: bias_row4 of n.
__device__ __forceinline__ v4f finish4(const GemmF32Args &g, v4f v, v4f row, int m, int n)
{
#pragma unroll
   for (int e = 0; e < 4; ++e) {
      v[e] = __fmul_rn(g.alpha, v[e]);
      if (g.bias_kind == SOFIE_BIAS_ROW) v[e] = __fadd_rn(v[e], __fmul_rn(g.beta, row[e]));
      else if (g.bias_kind == SOFIE_BIAS_FULL && n + e < g.N) v[e] = __fadd_rn(v[e], __fmul_rn(g.beta, g.bias[(size_t)m * g.ldy + n + e]));
      else if (g.bias_kind == SOFIE_BIAS_COL) v[e] = __fadd_rn(v[e], __fmul_rn(g.beta, g.bias[m]));
      if (g.relu) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
   }
   return v;
}
__device__ __forceinline__ void store4(const GemmF32Args &g, v4f v, int m, int n)
{
   float *o = g.Y + (size_t)m * g.ldy + n;
   if (n + 4 <= g.N) {
      __builtin_memcpy(o, &v, 16);       // rows may start on any float
      return;
   }
#pragma unroll
   for (int e = 0; e < 3; ++e)
      if (n + e < g.N) o[e] = v[e];
}
// The last four columns of all, of which those in front of `first` are stored by whoever's sums of them may have been formed in another way.
__device__ __forceinline__ void store4_from(const GemmF32Args &g, v4f v, int m, int n, int first)
{
   if (n >= first) return store4(g, v, m, n);
   float *o = g.Y + (size_t)m * g.ldy + n;
#pragma unroll
   for (int e = 1; e < 4; ++e)
      if (n + e >= first) o[e] = v[e];
}

// k_gemm_f32_split (gemm_f32_split.hip): the product on the bf16 matrix instructions, operands as three bf16 numbers, 16 mi rows x 64
// columns per workgroup, K in `splits` slices (above one: raw sums into g.partial, for k_gemm_f32_skinny_finish).
struct SplitChoice {
   int mi, splits;
   float us;
};
// The form with the shortest estimate; us = 1e30 where the kernel does not take the product. mi = 8 (gemm_f32_shared_choice): tiles of 128 x 128 whose
// operands are split once for all wavefronts.
SplitChoice gemm_f32_split_choice(const sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, bool one_launch);
SplitChoice gemm_f32_shared_choice(const sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz);
int launch_gemm_f32_split(sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, const SplitChoice &c);

}  // namespace sofie
