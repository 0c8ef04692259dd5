// fp32 GEMM on the matrix cores with a fused alpha / beta*bias / ReLU epilogue: k_gemm_f32_dma (v_mfma_f32_32x32x2_f32) for
// operands that can be fetched 16 bytes at a time, k_gemm_f32 (v_mfma_f32_16x16x4_f32) for all others, k_gemm_f32_skinny for
// few rows; k_gemm_f32_split (gemm_f32_split.hip) where its estimate is the shortest. Roofline: MFMA fp32 (256 flop/clk/CU).
#include <cstdint>
#include <type_traits>

#include "common.h"
#include "gemm_tile.h"
#include "gemm_f32.h"
#include "gemm_f32_operand.h"

using namespace sofie;

namespace {

// Products of any sizes, leading dimensions and storage (A_KM: A stored [K][M], B_KM: B stored [K][N]). 256 threads = 4
// wavefronts in 2 x 2, each with MI x NJ tiles of 16 x 16 (v_mfma_f32_16x16x4_f32: tiles of 16 let a product take workgroup
// tiles of 32 to 128 rows and columns, so that their number suits the device: 1500 x 1001 is 256 tiles of 96 x 64). Both
// operand tiles travel global memory -> LDS without registers, 16 bytes per lane (buffer_load_dwordx4 ... lds, which takes any
// address on a dword; 4 bytes per lane cost the same time per request, 33 cycles of a compute unit), in 2 or 3 stages of 32 k:
//   * inside 16 k lane group kg (lane / 16) supplies k = 4 kg + e to matrix instruction e;
//   * an operand with rows along K lies in rows of 8 chunks of 16 bytes, chunk c of row r in slot c ^ ((r >> 1) & 7): the 16
//     rows a lane group reads with one 16-byte read per lane fall on 16 slots;
//   * an operand with rows along M or N lies in rows of k, rotated by 16 columns per four k (one 4-byte read per
//     instruction, the lane groups on different banks).
// Cells outside the matrices ask for an offset outside the descriptor and arrive as zeros, or, behind M and N, hold
// what lies there and are not stored. Only where a 16-byte piece would straddle the end of K (rows along K) or of the
// whole matrix (rows along N, last row) the last step travels 4 bytes per lane (F32Operand). Bound: fp32 matrix instructions.

// Registers of a lane's reads of one operand tile: T tiles of 16 rows (columns) from `first` on.
template <bool KM, int ROWS, int T>
struct F32Fragments {
   int at[KM ? T : 2];
   __device__ __forceinline__ void init(int first, int r16, int kg)
   {
      if constexpr (KM) {
#pragma unroll
         for (int t = 0; t < T; ++t) at[t] = 4 * kg * ROWS + (first + t * 16 + 16 * kg) % ROWS + r16;
      } else {
#pragma unroll
         for (int s = 0; s < 2; ++s) at[s] = (first + r16) * 32 + (((s * 4 + kg) ^ ((r16 >> 1) & 7)) << 2);
      }
   }
   __device__ __forceinline__ v4f read(const float *tile, int s, int t) const
   {
      if constexpr (KM) {
         v4f f;
#pragma unroll
         for (int e = 0; e < 4; ++e) f[e] = tile[at[t] + (s * 16 + e) * ROWS];
         return f;
      } else {
         return *reinterpret_cast<const v4f *>(tile + at[s] + t * 16 * 32);
      }
   }
};

template <bool A_KM, bool B_KM, int MI, int NJ>
__global__ void __launch_bounds__(256, MI * NJ >= 9 ? 2 : 3) k_gemm_f32(GemmF32Args g)
{
   constexpr int BM = 32 * MI, BN = 32 * NJ, BK = 32, STAGE = (BM + BN) * BK;
   constexpr int NST = BM + BN > 192 ? 2 : 3;
   constexpr int RQ = F32Operand<A_KM, BM>::NRQ + F32Operand<B_KM, BN>::NRQ;      // requests per wavefront and stage, at least
   extern __shared__ __align__(16) unsigned char smem_raw[];
   float *const lds = reinterpret_cast<float *>(smem_raw);
   const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw;
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, kg = lane >> 4;
   if (g.n_lead > 0) select_product(g, (long long)blockIdx.z + g.z0);
   int tm, tn;
   tile_of(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
   const int m0 = tm * BM, n0 = tn * BN;
   int kt_begin = 0, kt_end = (g.K + BK - 1) / BK;
   if (gridDim.y > 1) {      // K in slices: raw sums into the slice's plane of the scratch buffer
      const int per = (kt_end + (int)gridDim.y - 1) / (int)gridDim.y;
      kt_begin = (int)blockIdx.y * per;
      kt_end = kt_end < kt_begin + per ? kt_end : kt_begin + per;
      g.Y = g.partial + (size_t)blockIdx.y * g.M * g.N;
      g.ldy = g.N;
      g.alpha = 1.0f;
      g.bias_kind = SOFIE_BIAS_NONE;
      g.relu = 0;
   }
   F32Operand<A_KM, BM> oa;
   F32Operand<B_KM, BN> ob;
   oa.init(g.A, g.lda, m0, g.M, g.K, tid);
   ob.init(g.B, g.ldb, n0, g.N, g.K, tid);
   F32Fragments<A_KM, BM, MI> ra;
   F32Fragments<B_KM, BN, NJ> rb;
   ra.init(wm * 16 * MI, r16, kg);
   rb.init(wn * 16 * NJ, r16, kg);
   v4f row[NJ];
#pragma unroll
   for (int j = 0; j < NJ; ++j) row[j] = bias_row4(g, n0 + wn * 16 * NJ + j * 16 + kg * 4);
   v4f acc[MI][NJ];
#pragma unroll
   for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
   auto request = [&](auto whole, int kt, int stage) {
      // (a step behind the last one is requested again with nothing in it, so that the waits count the same requests)
      const unsigned dst = lds0 + (unsigned)(stage * STAGE * 4);
      oa.template request<decltype(whole)::value>(kt, dst, wave);
      ob.template request<decltype(whole)::value>(kt, dst + BM * BK * 4, wave);
   };
   auto multiply = [&](const float *tile) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
         v4f fa[MI], fb[NJ];
#pragma unroll
         for (int i = 0; i < MI; ++i) fa[i] = ra.read(tile, s, i);
#pragma unroll
         for (int j = 0; j < NJ; ++j) fb[j] = rb.read(tile + BM * BK, s, j);
         // rows of the result tile are columns n (the B operand first): a lane ends up with 4 consecutive columns of a row
#pragma unroll
         for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
               for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][e], fa[i][e], acc[i][j], 0, 0, 0);
      }
   };
#pragma unroll
   for (int d = 0; d < NST - 1; ++d) request(std::false_type{}, kt_begin + d, d);
   int kt = kt_begin;
   // steps that need no check (of the requests, which are NST - 1 steps ahead), then the others
   const int whole_a = oa.whole_steps(), whole_b = ob.whole_steps(), whole_ab = whole_a < whole_b ? whole_a : whole_b;
   const int whole_steps = whole_ab < kt_end ? whole_ab : kt_end;
   for (; kt + 2 * NST - 2 < whole_steps; kt += NST) {
#pragma unroll
      for (int d = 0; d < NST; ++d) {
         wait_vmcnt<(NST - 2) * RQ>();
         __syncthreads();      // stage d has landed for every wavefront, and everybody is done with the one in front of it
         request(std::true_type{}, kt + d + NST - 1, (d + NST - 1) % NST);
         multiply(lds + d * STAGE);
      }
   }
   for (; kt < kt_end; kt += NST) {
#pragma unroll
      for (int d = 0; d < NST; ++d) {
         if (kt + d >= kt_end) break;
         wait_vmcnt<(NST - 2) * RQ>();
         __syncthreads();
         request(std::false_type{}, kt + d + NST - 1, (d + NST - 1) % NST);
         multiply(lds + d * STAGE);
      }
   }
   wait_vmcnt<0>();            // requests of stages nobody reads may not outlive the workgroup
#pragma unroll
   for (int i = 0; i < MI; ++i) {
      const int m = m0 + wm * 16 * MI + i * 16 + r16;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
         const int n = n0 + wn * 16 * NJ + j * 16 + kg * 4;
         if (m < g.M && n < g.N) store4(g, finish4(g, acc[i][j], row[j], m, n), m, n);
      }
   }
}

// The same product for operands that allow it (A [M][K] row-major, K a multiple of 32, 16-byte aligned rows), with
// both operand tiles travelling global memory -> LDS without registers (buffer_load_dwordx4 ... lds), two stages of
// 32 k, under the matrix loop of the stage before. Tile of 64 T x 64 T (T = 2: 128 x 128, two workgroups per CU; T = 1
// for products of few tiles: 64 x 64, four per CU), 4 wavefronts of T x T tiles of 32 x 32.
//   * An operand whose rows run along K (A; B given [N][K]) is staged as rows of 32 floats (8 chunks of 16 bytes) with
//     chunk c of row r in slot c ^ ((r >> 1) & 7): a lane reads 4 consecutive k of its row with one 16-byte read (lanes
//     0-31: k = 8s .. 8s+3, lanes 32-63: k = 8s+4 .. 8s+7, which is the pairing of four matrix instructions), and the 16
//     lanes the LDS serves together fall on 16 different slots of 256 bytes. The swizzle costs nothing: a lane of the
//     request asks for the chunk that belongs into its slot.
//   * B given [K][N] is staged as it is, rows of k with the tile's columns, and read 4 bytes per lane.
// A lane's read addresses do not depend on the K step (the stage is an immediate offset: the loop is unrolled over the
// two stages), so the loop holds LDS reads and matrix instructions and no vector arithmetic, which would take issue
// cycles from the matrix instructions. Rows behind M (or N) lie outside the tile's descriptor and arrive as zeros;
// outputs go through a descriptor too (columns behind N get an offset outside it and are dropped).
template <bool B_KMAJOR, int T>
__global__ void __launch_bounds__(256, T == 2 ? 2 : 4) k_gemm_f32_dma(GemmF32Args g)
{
   constexpr int BM = 64 * T, BN = 64 * T, BKD = 32;
   constexpr int STAGE = (BM + BN) * BKD;               // floats of one stage: the A tile, then the B tile
   constexpr unsigned OUTSIDE = 0x80000000u;            // an offset no descriptor of this kernel reaches
   extern __shared__ __align__(16) unsigned char smem_raw[];
   float *const lds = reinterpret_cast<float *>(smem_raw);
   const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw;
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int wm = wave >> 1, wn = wave & 1;
   const int fr = lane & 31, fk = lane >> 5;
   int tm, tn;
   tile_of(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
   const int m0 = tm * BM, n0 = tn * BN;
   const int rows_a = g.M - m0 < BM ? g.M - m0 : BM, rows_b = g.N - n0 < BN ? g.N - n0 : BN;
   // K in slices (few tiles, long K): this workgroup's steps of 32 k, raw sums into its plane of the scratch buffer
   int kt_begin = 0, kt_end = g.K / BKD;
   if (gridDim.y > 1) {
      const int per = (kt_end + (int)gridDim.y - 1) / (int)gridDim.y;
      kt_begin = (int)blockIdx.y * per;
      kt_end = kt_end < kt_begin + per ? kt_end : kt_begin + per;
      g.Y = g.partial + (size_t)blockIdx.y * g.M * g.N;
      g.ldy = g.N;
      g.alpha = 1.0f;
      g.bias_kind = SOFIE_BIAS_NONE;
      g.relu = 0;
   }
   const rsrc_t ars = make_rsrc(g.A + (size_t)m0 * g.lda, (unsigned)((size_t)rows_a * g.lda * 4));
   const rsrc_t brs = B_KMAJOR ? make_rsrc(g.B, (unsigned)((size_t)g.K * g.ldb * 4))
                               : make_rsrc(g.B + (size_t)n0 * g.ldb, (unsigned)((size_t)rows_b * g.ldb * 4));
   // requests: 16 bytes per lane, 256 lanes per request. Row-major operand: lane -> (row tid/8 [+ 32 per request],
   // slot tid%8), it fetches chunk slot ^ swizzle(row); the swizzle is the same for every request of the lane.
   constexpr int NRQ = 2 * T;                           // requests per operand tile and stage (4 KB each)
   const int rq_row = tid >> 3, rq_slot = tid & 7;
   const unsigned rq_a = (unsigned)((rq_row * g.lda + ((rq_slot ^ ((rq_row >> 1) & 7)) << 2)) * 4);
   unsigned rq_b;
   if constexpr (B_KMAJOR) {
      // lane -> (k tid/(BN/4) [+ 1024/BN per request], columns 4*(tid%(BN/4)) .. +3); columns behind N ask for nothing
      const int col = n0 + (tid % (BN / 4)) * 4;
      rq_b = col < g.N ? (unsigned)(((tid / (BN / 4)) * g.ldb + col) * 4) : OUTSIDE;
   } else {
      rq_b = (unsigned)((rq_row * g.ldb + ((rq_slot ^ ((rq_row >> 1) & 7)) << 2)) * 4);
   }
   const unsigned step_a = (unsigned)(32 * g.lda * 4), step_b = (unsigned)((B_KMAJOR ? 1024 / BN : 32) * g.ldb * 4);
   auto request = [&](int kt, int stage) {
      const unsigned dst = lds0 + (unsigned)(stage * STAGE * 4) + (unsigned)(wave * 1024);
      const unsigned ka = (unsigned)(kt * BKD * 4), kb = B_KMAJOR ? (unsigned)kt * BKD * (unsigned)g.ldb * 4u : ka;
#pragma unroll
      for (int u = 0; u < NRQ; ++u) dma16(ars, dst + u * 4096, (int)rq_a, (int)(ka + u * step_a));
#pragma unroll
      for (int u = 0; u < NRQ; ++u) dma16(brs, dst + BM * BKD * 4 + u * 4096, (int)rq_b, (int)(kb + u * step_b));
   };
   // read addresses of the lane's fragments in stage 0 (floats from the start of the LDS block)
   int ra[T][4], rb[T][4];
#pragma unroll
   for (int i = 0; i < T; ++i) {
      const int row = wm * 32 * T + i * 32 + fr;
#pragma unroll
      for (int s = 0; s < 4; ++s) ra[i][s] = row * BKD + (((2 * s + fk) ^ ((row >> 1) & 7)) << 2);
   }
#pragma unroll
   for (int j = 0; j < T; ++j) {
      const int row = wn * 32 * T + j * 32 + fr;
#pragma unroll
      for (int s = 0; s < 4; ++s)
         rb[j][s] = BM * BKD + (B_KMAJOR ? (8 * s + 4 * fk) * BN + row : row * BKD + (((2 * s + fk) ^ ((row >> 1) & 7)) << 2));
   }
   v16f acc[T][T];
#pragma unroll
   for (int i = 0; i < T; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j)
#pragma unroll
         for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

   auto multiply = [&](auto stage_c) {
      constexpr int OFF = decltype(stage_c)::value * STAGE;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
         v4f fa[T], fb[T];
#pragma unroll
         for (int i = 0; i < T; ++i) fa[i] = *reinterpret_cast<const v4f *>(lds + OFF + ra[i][s]);
#pragma unroll
         for (int j = 0; j < T; ++j) {
            if constexpr (B_KMAJOR) {
#pragma unroll
               for (int e = 0; e < 4; ++e) fb[j][e] = lds[OFF + rb[j][s] + e * BN];
            } else {
               fb[j] = *reinterpret_cast<const v4f *>(lds + OFF + rb[j][s]);
            }
         }
#pragma unroll
         for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
               for (int j = 0; j < T; ++j)
                  acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][e], fb[j][e], acc[i][j], 0, 0, 0);
      }
   };
   const int nk = kt_end;
   if (kt_begin < nk) request(kt_begin, 0);
   wait_vmcnt<0>();
   __syncthreads();
   for (int kt = kt_begin; kt < nk; kt += 2) {
      if (kt + 1 < nk) request(kt + 1, 1);
      multiply(std::integral_constant<int, 0>{});
      wait_vmcnt<0>();
      __syncthreads();        // stage 1 has landed, everybody is done with stage 0
      if (kt + 1 >= nk) break;
      if (kt + 2 < nk) request(kt + 2, 0);
      multiply(std::integral_constant<int, 1>{});
      wait_vmcnt<0>();
      __syncthreads();
   }

   // epilogue: v = alpha * acc (+ beta * bias) (ReLU); a lane holds column n = fr of 16 rows per tile
   const rsrc_t yrs = make_rsrc(g.Y + (size_t)m0 * g.ldy, (unsigned)((size_t)rows_a * g.ldy * 4));
   const __amdgpu_buffer_rsrc_t col_bias = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(g.bias) + (g.bias_kind == SOFIE_BIAS_COL ? m0 : 0), 0, g.bias_kind == SOFIE_BIAS_COL ? rows_a * 4 : 0, 0x00020000);
   const unsigned ldy4 = (unsigned)g.ldy * 4u;
#pragma unroll
   for (int j = 0; j < T; ++j) {
      const int n = n0 + wn * 32 * T + j * 32 + fr;
      const float brow = g.bias_kind == SOFIE_BIAS_ROW && n < g.N ? __fmul_rn(g.beta, g.bias[n]) : 0.0f;
      const unsigned voff = n < g.N ? (unsigned)(n * 4) + (unsigned)fk * 4u * ldy4 : OUTSIDE;
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
         for (int r = 0; r < 16; ++r) {
            const int m_uniform = wm * 32 * T + i * 32 + (r >> 2) * 8 + (r & 3);      // + 4 * fk in the lane's offset
            float v = __fmul_rn(g.alpha, acc[i][j][r]);
            if (g.bias_kind == SOFIE_BIAS_ROW) v = __fadd_rn(v, brow);
            else if (g.bias_kind == SOFIE_BIAS_COL)
               v = __fadd_rn(v, __fmul_rn(g.beta, __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(col_bias, fk * 16, m_uniform * 4, 0))));
            if (g.relu) v = v > 0.0f ? v : 0.0f;
            store4_buf(yrs, v, voff, (unsigned)m_uniform * ldy4);
         }
   }
}

// Small products of any storage and alignment: a workgroup owns 16 MI rows x 16 NJ columns and all of K. Its eight
// wavefronts take the chunks of 32 k in turn, DEPTH chunks of loads in flight each, straight from global memory into the
// operand registers (lane group kg supplies k = 8 kg + e of a chunk to instruction e), no LDS and no barrier on the way;
// their sums meet in LDS in a fixed order. A product this small is latency: one trip to memory, where the tiled kernel makes
// one per K-step and the products with K in slices launch twice.
template <bool A_KM, bool B_KM, int MI, int NJ>
__global__ void __launch_bounds__(512, MI * NJ == 4 ? 2 : 4) k_gemm_f32_direct(GemmF32Args g)
{
   constexpr int CH = 32, STEP = 8 * CH;
   constexpr int DEPTH = MI * NJ == 1 ? 3 : 2;
   constexpr int V = MI * NJ * 64;                     // quads of output columns of the tile
   __shared__ __align__(16) v4f red[8][V];
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int r16 = lane & 15, kg = lane >> 4;
   if (g.n_lead > 0) select_product(g, (long long)blockIdx.z + g.z0);
   int tm, tn;
   tile_of(blockIdx.x, (g.M + 16 * MI - 1) / (16 * MI), (g.N + 16 * NJ - 1) / (16 * NJ), tm, tn);
   const int m0 = tm * 16 * MI, n0 = tn * 16 * NJ;
   // rows and columns behind the matrix are copies of the last one; their results are not stored
   const float *pa[MI], *pb[NJ];
#pragma unroll
   for (int i = 0; i < MI; ++i) {
      const int m = m0 + i * 16 + r16 < g.M ? m0 + i * 16 + r16 : g.M - 1;
      pa[i] = A_KM ? g.A + m : g.A + (size_t)m * g.lda;
   }
#pragma unroll
   for (int j = 0; j < NJ; ++j) {
      const int n = n0 + j * 16 + r16 < g.N ? n0 + j * 16 + r16 : g.N - 1;
      pb[j] = B_KM ? g.B + n : g.B + (size_t)n * g.ldb;
   }
   struct Chunk {
      v4f a[MI][2], b[NJ][2];
   };
   // the outputs this thread will finish
   const int m = m0 + (tid / (64 * NJ)) * 16 + (tid & 15), n = n0 + (tid / 64 % NJ) * 16 + ((tid >> 4) & 3) * 4;
   const v4f bias = tid < V ? bias_row4(g, n) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
   // every load stays inside its row (column): the last ones are moved down to end with it
   auto fetch = [&](v4f &v, const float *p, int ld, bool km, int k) {
      if (km) {
#pragma unroll
         for (int e = 0; e < 4; ++e) v[e] = p[(size_t)(k + e < g.K ? k + e : g.K - 1) * ld];
      } else {
         __builtin_memcpy(&v, p + (k < g.K - 4 ? k : g.K - 4), 16);
      }
   };
   auto load = [&](Chunk &c, int k0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
         for (int i = 0; i < MI; ++i) fetch(c.a[i][h], pa[i], g.lda, A_KM, k0 + kg * 8 + h * 4);
#pragma unroll
         for (int j = 0; j < NJ; ++j) fetch(c.b[j][h], pb[j], g.ldb, B_KM, k0 + kg * 8 + h * 4);
      }
   };
   // two sums per output: shorter chains of rounded additions (relative error of two layers of 1024 1.6e-7 -> 1.25e-7) that do
   // not wait for each other (four layers of 300 on 16 rows 17.8 -> 16.1 us)
   v4f acc[2][MI][NJ];
#pragma unroll
   for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[0][i][j] = acc[1][i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
   // values of k .. k + 3 out of a load that may have been moved down, zero behind K
   auto trim = [&](v4f v, bool km, int k) {
      const int drop = km ? 0 : k - (g.K - 4);
      v4f r = v;
      if (drop > 0) {
         if (drop & 1) r = v4f{r[1], r[2], r[3], 0.0f};
         if (drop & 2) r = v4f{r[2], r[3], 0.0f, 0.0f};
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = k + e < g.K ? r[e] : 0.0f;
      return r;
   };
   auto multiply = [&](Chunk &c, int k0) {
      if (k0 + CH > g.K) {      // uniform: the last chunk
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const int k = k0 + kg * 8 + h * 4;
#pragma unroll
            for (int i = 0; i < MI; ++i) c.a[i][h] = trim(c.a[i][h], A_KM, k);
#pragma unroll
            for (int j = 0; j < NJ; ++j) c.b[j][h] = trim(c.b[j][h], B_KM, k);
         }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
         for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
               for (int j = 0; j < NJ; ++j) acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(c.b[j][h][e], c.a[i][h][e], acc[h][i][j], 0, 0, 0);
   };
   Chunk c[DEPTH];
   int k0 = wave * CH;
#pragma unroll
   for (int d = 0; d < DEPTH; ++d) load(c[d], k0 + d * STEP);
   while (k0 < g.K) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
         if (k0 < g.K) multiply(c[d], k0);
         if (k0 + DEPTH * STEP < g.K) load(c[d], k0 + DEPTH * STEP);
         k0 += STEP;
      }
   }
#pragma unroll
   for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) red[wave][(i * NJ + j) * 64 + lane] = acc[0][i][j] + acc[1][i][j];
   __syncthreads();
   if (tid >= V || m >= g.M || n >= g.N) return;
   v4f s = red[0][tid];
#pragma unroll
   for (int w = 1; w < 8; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = __fadd_rn(s[e], red[w][tid][e]);
   store4(g, finish4(g, s, bias, m, n), m, n);
}

// One thread per output: K below the eight where operands would be shared, on rows of millions of floats.
__global__ void __launch_bounds__(256) k_gemm_f32_plain(GemmF32Args g)
{
   const size_t idx = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
   if (idx >= (size_t)g.M * g.N) return;
   if (g.n_lead > 0) select_product(g, (long long)blockIdx.z + g.z0);
   const int m = (int)(idx / g.N), n = (int)(idx % g.N);
   float v = 0.0f;
   for (int k = 0; k < g.K; ++k)
      v = fmaf(g.transA ? g.A[(size_t)k * g.lda + m] : g.A[(size_t)m * g.lda + k], g.transB ? g.B[(size_t)n * g.ldb + k] : g.B[(size_t)k * g.ldb + n], v);
   v = __fmul_rn(g.alpha, v);
   if (g.bias_kind == SOFIE_BIAS_ROW) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[n]));
   else if (g.bias_kind == SOFIE_BIAS_FULL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[(size_t)m * g.ldy + n]));
   else if (g.bias_kind == SOFIE_BIAS_COL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[m]));
   if (g.relu) v = v > 0.0f ? v : 0.0f;
   g.Y[(size_t)m * g.ldy + n] = v;
}

// Few rows of A (M <= 64: a layer on a small batch): the product is a pass over B, bound by memory, and tiles of
// 64 x 64 outputs would leave most of the device idle. Here a wavefront owns all rows of A (MT tiles of T = 16 rows,
// v_mfma_f32_16x16x4_f32) and 4 T = 64 columns: its accumulators are MT x 4 tiles of T x T (rows of A x columns), and B
// goes from global memory straight into the matrix instructions' operand registers, 16 bytes per lane, with no LDS on
// the way. With lane = (j = lane % T, kg = lane / T):
//   * B [K][N]: a lane loads columns 4 j .. 4 j + 3 of row k0 + 4 kg + u (a wavefront's load: 4 rows of 256
//     contiguous bytes); element e of the four feeds the tile of columns 4 j + e, so a lane ends up with 4 consecutive
//     columns of a row.
//   * B [N][K]: a lane loads k0 + 4 kg .. + 3 of column T q + j; element u feeds instruction u of tile q.
// A lane's 4 consecutive k of its row of A arrive the same way (k0 + 4 kg .. + 3, one instruction per element). The
// grid is column blocks x slices of K; the four wavefronts of a workgroup take the slice's chunks of 16 k in turn,
// each with the loads of the next three chunks in flight while it multiplies, and add their accumulators up through
// LDS. With more than one slice the sums go to a scratch buffer [slice][M][N] and k_gemm_f32_skinny_finish adds them
// in slice order and applies alpha, bias and ReLU (a fixed order: the result does not depend on timing). Rows behind
// M, columns behind N and k behind the slice get offsets outside the buffer descriptors and arrive as zeros.
template <int T> struct SkinnyTile;
template <> struct SkinnyTile<16> {
   typedef v4f Acc;
   static constexpr int NR = 4;
   static __device__ __forceinline__ Acc mma(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
   static __device__ __forceinline__ int row(int r, int kg) { return kg * 4 + r; }
};

template <bool B_NK, int T, int MT>
__global__ void __launch_bounds__(256) k_gemm_f32_skinny(GemmF32Args g, float *partial, int kslice, int splits)
{
   typedef SkinnyTile<T> Tile;
   constexpr int NR = Tile::NR;
   constexpr int CHUNK = 256 / T;                      // k per chunk: 4 per lane, 64 / T groups of lanes
   constexpr int COLS = 4 * T;                         // columns of a workgroup
   constexpr unsigned OUTSIDE = 0x80000000u;
   __shared__ float red[2 * MT * 4 * NR * 64];
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int fr = lane % T, fk = lane / T;
   const int c0 = blockIdx.x * COLS;
   const int k_begin = blockIdx.y * kslice;
   const int k_end = g.K < k_begin + kslice ? g.K : k_begin + kslice;
   const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(g.A), 0, (int)(((size_t)(g.M - 1) * g.lda + g.K) * 4), 0x00020000);
   const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(g.B), 0, (int)((B_NK ? (size_t)(g.N - 1) * g.ldb + g.K : (size_t)(g.K - 1) * g.ldb + g.N) * 4), 0x00020000);
   unsigned a_off[MT], b_off[B_NK ? 4 : 1];
#pragma unroll
   for (int t = 0; t < MT; ++t) a_off[t] = t * T + fr < g.M ? (unsigned)(((t * T + fr) * g.lda + 4 * fk) * 4) : OUTSIDE;
   if constexpr (B_NK) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
         const int n = c0 + T * q + fr;
         b_off[q] = n < g.N ? (unsigned)((n * g.ldb + 4 * fk) * 4) : OUTSIDE;
      }
   } else {
      const int n = c0 + 4 * fr;
      b_off[0] = n < g.N ? (unsigned)((4 * fk * g.ldb + n) * 4) : OUTSIDE;
   }
   struct Chunk {
      v4f a[MT], b[4];
   };
   auto load = [&](Chunk &c, int k0) {
      // a lane's four k lie inside the slice together or not at all (K and the slices are multiples of 4)
      const bool in = k0 + 4 * fk < k_end;
#pragma unroll
      for (int t = 0; t < MT; ++t)
         c.a[t] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(ars, in ? a_off[t] : OUTSIDE, k0 * 4, 0));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
         if constexpr (B_NK)
            c.b[q] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(brs, in ? b_off[q] : OUTSIDE, k0 * 4, 0));
         else
            c.b[q] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(brs, in ? b_off[0] : OUTSIDE, (k0 + q) * g.ldb * 4, 0));
      }
   };
   typename Tile::Acc acc[MT][4];
#pragma unroll
   for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
         for (int r = 0; r < NR; ++r) acc[t][q][r] = 0.0f;
   auto multiply = [&](const Chunk &c) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
         for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
               // B [K][N]: load u is row k0 + 4 kg + u, its element q a column; B [N][K]: load q is a group of columns,
               // its element u a k
               const float b = B_NK ? c.b[q][u] : c.b[u][q];
               acc[t][q] = Tile::mma(c.a[t][u], b, acc[t][q]);
            }
   };
   // chunks wave, wave + 4, ... of the slice; three chunks ahead are in flight while one is multiplied (loads behind
   // the slice's end ask for nothing)
   constexpr int STEP = 4 * CHUNK;
   Chunk c0_, c1_, c2_, c3_;
   int k0 = k_begin + wave * CHUNK;
   load(c0_, k0);
   load(c1_, k0 + STEP);
   load(c2_, k0 + 2 * STEP);
   // the bias of the lane's four columns, requested behind the first operands and ahead of the loop, which does not wait for it (one
   // load per output behind the loop was most of a short product's time: 52 x 1113 x 184 17.6 us; beta * bias in front of it
   // cost 0.6 us, also where a slice has no use for it: 2 x 192 x 5828 8.7 against 7.8 us)
   const bool last = splits == 1;
   float brow[4];
#pragma unroll
   for (int q = 0; q < 4; ++q) {
      const int n = B_NK ? c0 + T * q + fr : c0 + 4 * fr + q;
      brow[q] = last && g.bias_kind == SOFIE_BIAS_ROW && n < g.N ? g.bias[n] : 0.0f;
   }
   for (; k0 < k_end; k0 += STEP) {
      load(c3_, k0 + 3 * STEP);
      multiply(c0_);
      c0_ = c1_;
      c1_ = c2_;
      c2_ = c3_;
   }
   // the four wavefronts' sums meet in LDS: wavefronts 2 and 3 hand theirs to 0 and 1, then 1 hands its to 0
   // ((w0 + w2) + (w1 + w3): a fixed order)
   auto put = [&](float *dst) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
         for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < NR; ++r) dst[((t * 4 + q) * NR + r) * 64 + lane] = acc[t][q][r];
   };
   auto add = [&](const float *src) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
         for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[t][q][r] = __fadd_rn(acc[t][q][r], src[((t * 4 + q) * NR + r) * 64 + lane]);
   };
   constexpr int BLOCK = MT * 4 * NR * 64;
   if (wave >= 2) put(red + (wave - 2) * BLOCK);
   __syncthreads();
   if (wave < 2) add(red + wave * BLOCK);
   __syncthreads();
   if (wave == 1) put(red);
   __syncthreads();
   if (wave == 0) add(red);
   if (wave != 0) return;
   // tile (t, q), register r of a lane: row t * T + Tile::row(r, kg); column c0 + 4 j + q (B [K][N]) or c0 + T q + j
   float *const out = last ? g.Y : partial + (size_t)blockIdx.y * g.M * g.N;
   const int ldo = last ? g.ldy : g.N;
   const bool vec_out = !last || (g.ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(g.Y) & 15u) == 0);   // rows of whole 16-byte chunks
   auto finish = [&](float v, int q, int m, int n) {
      if (!last) return v;
      v = __fmul_rn(g.alpha, v);
      if (g.bias_kind == SOFIE_BIAS_ROW) v = __fadd_rn(v, __fmul_rn(g.beta, brow[q]));
      else if (g.bias_kind == SOFIE_BIAS_FULL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[(size_t)m * g.ldy + n]));
      else if (g.bias_kind == SOFIE_BIAS_COL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[m]));
      if (g.relu) v = v > 0.0f ? v : 0.0f;
      return v;
   };
#pragma unroll
   for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
         const int m = t * T + Tile::row(r, fk);
         if (m >= g.M) continue;
         if constexpr (B_NK) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
               const int n = c0 + T * q + fr;
               if (n < g.N) out[(size_t)m * ldo + n] = finish(acc[t][q][r], q, m, n);
            }
         } else {
            const int n = c0 + 4 * fr;     // N is a multiple of 4 on this path: the four columns are inside together
            if (n < g.N) {
               float *o = out + (size_t)m * ldo + n;
               const v4f v = {finish(acc[t][0][r], 0, m, n), finish(acc[t][1][r], 1, m, n + 1), finish(acc[t][2][r], 2, m, n + 2),
                              finish(acc[t][3][r], 3, m, n + 3)};
               if (vec_out) *reinterpret_cast<v4f *>(o) = v;
               else {
#pragma unroll
                  for (int q = 0; q < 4; ++q) o[q] = v[q];
               }
            }
         }
      }
}

// Sum of the K slices' partial products in slice order, then alpha, bias and ReLU: one thread per output. The loads of
// eight slices are in flight together; the additions keep the slices' order.
__global__ void __launch_bounds__(256) k_gemm_f32_skinny_finish(GemmF32Args g, const float *__restrict__ partial, int splits)
{
   ask_for_arguments<sizeof(g)>();
   const int idx = blockIdx.x * 256 + threadIdx.x;
   if (idx >= g.M * g.N) return;
   const int m = idx / g.N, n = idx - m * g.N;
   const size_t plane = (size_t)g.M * g.N;
   float v = 0.0f;
   int s = 0;
   for (; s + 8 <= splits; s += 8) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = partial[(size_t)(s + i) * plane + idx];
#pragma unroll
      for (int i = 0; i < 8; ++i) v = __fadd_rn(v, p[i]);
   }
   for (; s < splits; ++s) v = __fadd_rn(v, partial[(size_t)s * plane + idx]);
   v = __fmul_rn(g.alpha, v);
   if (g.bias_kind == SOFIE_BIAS_ROW) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[n]));
   else if (g.bias_kind == SOFIE_BIAS_FULL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[(size_t)m * g.ldy + n]));
   else if (g.bias_kind == SOFIE_BIAS_COL) v = __fadd_rn(v, __fmul_rn(g.beta, g.bias[m]));
   if (g.relu) v = v > 0.0f ? v : 0.0f;
   g.Y[(size_t)m * g.ldy + n] = v;
}

int launch_finish(sofie_hip_ctx *ctx, const GemmF32Args &g, int splits)
{
   hipLaunchKernelGGL(k_gemm_f32_skinny_finish, dim3(cdiv(g.M * g.N, 256)), dim3(256), 0, ctx->stream, g, g.partial, splits);
   return check_launch(ctx, "k_gemm_f32_skinny_finish");
}

// M <= 64 rows on k_gemm_f32_skinny. Slices of K so that about eight workgroups per compute unit exist, each wavefront
// with at least four chunks, and so that the partial sums stay below a quarter of B's bytes once they are more than a
// few megabytes (below that the launch is latency, not traffic).
template <bool B_NK, int T, int MT>
int launch_skinny_as(sofie_hip_ctx *ctx, GemmF32Args &g)
{
   constexpr int CHUNK = 256 / T;
   const int blocks = cdiv(g.N, 4 * T);
   int splits = 8 * ctx->num_cus / blocks;
   if (splits > g.K / (16 * CHUNK)) splits = g.K / (16 * CHUNK);
   if ((size_t)splits * g.M * g.N * 4 > ((size_t)4 << 20) && splits > g.K / (4 * g.M)) splits = g.K / (4 * g.M);
   if (splits < 1) splits = 1;
   const int kslice = cdiv(cdiv(g.K, splits), 4 * CHUNK) * 4 * CHUNK;
   splits = cdiv(g.K, kslice);
   float *partial = nullptr;
   if (splits > 1) {
      void *ws = nullptr;
      if (int rc = workspace(ctx, (size_t)splits * g.M * g.N * sizeof(float), &ws)) return rc;
      partial = static_cast<float *>(ws);
   }
   hipLaunchKernelGGL((k_gemm_f32_skinny<B_NK, T, MT>), dim3(blocks, splits), dim3(256), 0, ctx->stream, g, partial, kslice, splits);
   if (int rc = check_launch(ctx, "k_gemm_f32_skinny")) return rc;
   if (splits == 1) return SOFIE_HIP_OK;
   g.partial = partial;
   return launch_finish(ctx, g, splits);
}

int launch_skinny(sofie_hip_ctx *ctx, GemmF32Args &g)
{
   if (g.M <= 16) return g.transB ? launch_skinny_as<true, 16, 1>(ctx, g) : launch_skinny_as<false, 16, 1>(ctx, g);
   // 17 to 64 rows as two or four tiles of 16 rows: 32 x 32 tiles (twice the columns per wavefront, twice the
   // accumulator registers) measured 9 - 13 % slower (64 x 4096 x 4096: 42.7 against 37.7 us)
   if (g.M <= 32) return g.transB ? launch_skinny_as<true, 16, 2>(ctx, g) : launch_skinny_as<false, 16, 2>(ctx, g);
   return g.transB ? launch_skinny_as<true, 16, 4>(ctx, g) : launch_skinny_as<false, 16, 4>(ctx, g);
}

template <bool A_KM, bool B_KM, int MI, int NJ>
int launch_tiles_as(sofie_hip_ctx *ctx, GemmF32Args &g, int splits, unsigned nz)
{
   constexpr int BM = 32 * MI, BN = 32 * NJ, NST = BM + BN > 192 ? 2 : 3;
   constexpr auto kern = k_gemm_f32<A_KM, B_KM, MI, NJ>;
   SOFIE_LARGE_LDS(kern);
   hipLaunchKernelGGL(kern, dim3(cdiv(g.M, BM) * cdiv(g.N, BN), splits, nz), dim3(256), NST * (BM + BN) * 32 * 4, ctx->stream, g);
   if (int rc = check_launch(ctx, "k_gemm_f32")) return rc;
   if (splits == 1) return SOFIE_HIP_OK;
   return launch_finish(ctx, g, splits);
}

template <bool A_KM, bool B_KM, int MI, int NJ>
int launch_direct_as(sofie_hip_ctx *ctx, GemmF32Args &g, unsigned nz)
{
   hipLaunchKernelGGL((k_gemm_f32_direct<A_KM, B_KM, MI, NJ>), dim3(cdiv(g.M, 16 * MI) * cdiv(g.N, 16 * NJ), 1, nz), dim3(512), 0, ctx->stream, g);
   return check_launch(ctx, "k_gemm_f32_direct");
}

// The kernel for operands of any kind, by an estimate of its time behind the launch.
//   direct   1 us per round of resident workgroups, and the larger of its matrix instructions (550 GFLOP/s per compute unit) and
//            of what it reads (a compute unit takes in 43 bytes per ns)
//   tiles    the measured time of a K-step of 32, of a workgroup alone on its compute unit and of one among others (128 x 128:
//            1.95 / 1.91 us, of which 1.71 are its matrix instructions), and 2 us around it
//   slices   5 us for the pass that adds them, and their sums written and read at 6 TB/s
// Fitted to the times of every kernel on 34 sizes, 10 x 64 x 16 to 4000 x 4001 x 4002. Where the lines fall: 90 x 90 x 360 5.4 us
// direct, 6.4 on 32 x 32 tiles, 12.3 on 64 x 64; 1500 x 1001 x 1111 85 / 38 / 42, 34 on 32 x 64; 256 x 256 x 12800 39 direct, 90 on
// 32 x 32 tiles and 25 with them in 8 slices; 4000 x 4001 x 4002 978 on 64 x 64, 965 on 128 x 128.
enum GeneralKernel { TILES, DIRECT, SPLIT };
struct GeneralChoice {
   GeneralKernel kernel;
   int mi, nj, splits;
   float us;
};
constexpr int kDirectTiles[4][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}};
struct TileCost {
   int mi, nj;
   float alone, among;
};
constexpr TileCost kTileCosts[6] = {{1, 1, 0.21f, 0.176f}, {1, 2, 0.36f, 0.275f}, {2, 1, 0.36f, 0.275f}, {2, 2, 0.60f, 0.51f}, {3, 2, 0.85f, 0.78f}, {4, 4, 1.95f, 1.91f}};

// The tiled kernel's offsets are 32 bits wide: a K-step's 32 rows of an operand stored along M or N, a tile's rows of one along
// K. k_gemm_f32_direct takes any leading dimension. A launch holds fewer than 2^32 threads. us = 1e30: nothing fits (K below
// four on rows of 2^24 floats).
GeneralChoice general_choice(const sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, bool one_launch)
{
   GeneralChoice best = {TILES, 1, 1, 1, 1e30f};
   auto offsets_fit = [](bool km, int ld, int rows) { return (long long)(km ? 32 : rows) * ld * 4 < (1ll << 31); };
   const int cus = ctx->num_cus;
   auto consider = [&](GeneralKernel kernel, int mi, int nj, int splits, float us) {
      if (us < best.us) best = {kernel, mi, nj, splits, us};
   };
   auto consider_direct = [&] {
      for (const auto &t : kDirectTiles) {
         const int mi = t[0], nj = t[1], resident = mi * nj == 4 ? 1 : 2;
         const long long tiles = (long long)cdiv(g.M, 16 * mi) * cdiv(g.N, 16 * nj), per_cu = (tiles * nz + cus - 1) / cus;
         if (tiles >= (1ll << 32) / 512) continue;
         const float mfma = (float)per_cu * 512.0f * mi * nj * g.K / 550e3f, reads = (float)per_cu * 64.0f * (mi + nj) * g.K / 43e3f;
         consider(DIRECT, mi, nj, 1, 0.5f + (float)((per_cu + resident - 1) / resident) + (mfma > reads ? mfma : reads));
      }
   };
   if (g.K >= 4 && g.bias_kind != SOFIE_BIAS_FULL) consider_direct();
   const int steps = cdiv(g.K, 32);
   for (const auto &t : kTileCosts) {
      const long long tiles = (long long)cdiv(g.M, 32 * t.mi) * cdiv(g.N, 32 * t.nj) * nz;
      if (!offsets_fit(g.transA, g.lda, 32 * t.mi) || !offsets_fit(!g.transB, g.ldb, 32 * t.nj) || tiles / nz >= (1ll << 32) / 256) continue;
      for (int s = 1; s <= 16; s = s < 4 ? s + 1 : s * 2) {
         if (s > 1 && (one_launch || steps / s < 4 || (size_t)g.M * g.N >= ((size_t)1 << 28))) break;
         const long long per_cu = (tiles * s + cus - 1) / cus;
         const float step = per_cu == 1 ? t.alone : (float)per_cu * t.among;
         consider(TILES, t.mi, t.nj, s, 2.0f + step * cdiv(steps, s) + (s > 1 ? 5.0f + 8.0f * s * (float)g.M * g.N / 6e6f : 0.0f));
      }
   }
   // (operands as three bf16 numbers on the bf16 matrix instructions: 1500 x 1001 x 1111 29 us, 33 on 32 x 64 tiles)
   const SplitChoice split = gemm_f32_split_choice(ctx, g, nz, one_launch);
   consider(SPLIT, split.mi, 4, split.splits, split.us);
   // (in place of the fp32 instructions: 5938 x 7616 x 728, both transposed, 605 us, 423; 5776 x 1195 x 400 59, 49)
   if (best.kernel != SPLIT) {
      const SplitChoice shared = gemm_f32_shared_choice(ctx, g, nz);
      consider(SPLIT, shared.mi, 4, shared.splits, shared.us);
   }
   if (g.K >= 4 && best.us >= 1e30f) consider_direct();
   return best;
}

template <bool A_KM, bool B_KM>
int launch_general_as(sofie_hip_ctx *ctx, GemmF32Args &g, unsigned nz, const GeneralChoice &c)
{
   if (c.kernel == DIRECT) {
      switch (c.mi * 10 + c.nj) {
      case 11: return launch_direct_as<A_KM, B_KM, 1, 1>(ctx, g, nz);
      case 12: return launch_direct_as<A_KM, B_KM, 1, 2>(ctx, g, nz);
      case 21: return launch_direct_as<A_KM, B_KM, 2, 1>(ctx, g, nz);
      default: return launch_direct_as<A_KM, B_KM, 2, 2>(ctx, g, nz);
      }
   }
   switch (c.mi * 10 + c.nj) {
   case 11: return launch_tiles_as<A_KM, B_KM, 1, 1>(ctx, g, c.splits, nz);
   case 12: return launch_tiles_as<A_KM, B_KM, 1, 2>(ctx, g, c.splits, nz);
   case 21: return launch_tiles_as<A_KM, B_KM, 2, 1>(ctx, g, c.splits, nz);
   case 22: return launch_tiles_as<A_KM, B_KM, 2, 2>(ctx, g, c.splits, nz);
   case 32: return launch_tiles_as<A_KM, B_KM, 3, 2>(ctx, g, c.splits, nz);
   default: return launch_tiles_as<A_KM, B_KM, 4, 4>(ctx, g, c.splits, nz);
   }
}

// Operands of any size, alignment and storage; nz products of a stack (one_launch: K is not cut).
int launch_general(sofie_hip_ctx *ctx, GemmF32Args &g, unsigned nz, bool one_launch)
{
   GeneralChoice c = general_choice(ctx, g, nz, one_launch);
   if (c.splits > 1) {
      // without memory for the slices' sums (while a graph is recorded or alive) K stays in one piece
      g.partial = static_cast<float *>(workspace_if_room(ctx, (size_t)c.splits * g.M * g.N * sizeof(float)));
      if (!g.partial) c = general_choice(ctx, g, nz, true);
   }
   // a handful of k on rows of millions: a thread per output is the shortest way there (4194305 x 7 x 5: 161 us against
   // 264 on tiles)
   if (c.us >= 1e30f || (g.K < 8 && (g.lda >= (1 << 22) || g.ldb >= (1 << 22)))) {
      const size_t blocks = ((size_t)g.M * g.N + 255) / 256, across = blocks < ((size_t)1 << 23) ? blocks : (size_t)1 << 23;
      hipLaunchKernelGGL(k_gemm_f32_plain, dim3((unsigned)across, (unsigned)((blocks + across - 1) / across), nz), dim3(256), 0, ctx->stream, g);
      return check_launch(ctx, "k_gemm_f32_plain");
   }
   if (c.kernel == SPLIT) {
      if (int rc = launch_gemm_f32_split(ctx, g, nz, {c.mi, c.splits, c.us})) return rc;
      return c.splits > 1 ? launch_finish(ctx, g, c.splits) : SOFIE_HIP_OK;
   }
   if (g.transA) return g.transB ? launch_general_as<true, false>(ctx, g, nz, c) : launch_general_as<true, true>(ctx, g, nz, c);
   return g.transB ? launch_general_as<false, false>(ctx, g, nz, c) : launch_general_as<false, true>(ctx, g, nz, c);
}

}  // namespace

extern "C" int sofie_hip_gemm_f32(sofie_hip_ctx *ctx, int transA, int transB, int M, int N, int K, float alpha,
                                  const float *A, int lda, const float *B, int ldb, float beta, const float *bias,
                                  int bias_kind, float *Y, int ldy, int act)
{
   if (!ctx) return SOFIE_HIP_EINVAL;
   SOFIE_REQUIRE(ctx, M >= 0 && N >= 0 && K >= 0, "negative dimension");
   if (M == 0 || N == 0) return SOFIE_HIP_OK;
   SOFIE_REQUIRE(ctx, Y && (K == 0 || (A && B)), "null operand");
   SOFIE_REQUIRE(ctx, lda >= (transA ? M : K) && ldb >= (transB ? K : N) && ldy >= N, "leading dimension too small");
   SOFIE_REQUIRE(ctx, act == SOFIE_ACT_NONE || act == SOFIE_ACT_RELU, "unknown activation");
   SOFIE_REQUIRE(ctx, bias_kind >= SOFIE_BIAS_NONE && bias_kind <= SOFIE_BIAS_COL, "unknown bias kind");
   if (!bias || bias_kind == SOFIE_BIAS_NONE) {
      // Same rule as the reference emitter: without a bias tensor beta must be zero.
      if (beta != 0.0f)
         return sofie::set_error(ctx, SOFIE_HIP_EINVAL,
                                 "sofie_hip_gemm_f32: Bias tensor is not present but beta value in Gemm is not zero");
      bias = nullptr;
      bias_kind = SOFIE_BIAS_NONE;
   }
   GemmF32Args g{};
   g.A = A; g.B = B; g.bias = bias; g.Y = Y;
   g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldb = ldb; g.ldy = ldy;
   g.transA = transA != 0; g.transB = transB != 0;
   g.alpha = alpha; g.beta = beta; g.bias_kind = bias_kind; g.relu = act == SOFIE_ACT_RELU;
   const bool small = (size_t)cdiv(M, 128) * cdiv(N, 128) < 256;
   // operands by LDS-DMA: A row-major with rows of whole 16-byte chunks, K in whole stages, everything a descriptor
   // addresses below 2 GiB, a bias that is a row, a column or absent; 64 x 64 tiles where 128 x 128 ones would leave
   // compute units without a tile, and nothing for products of a handful of tiles
   const auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
   const int tile = small ? 64 : 128;
   const bool dma = (size_t)cdiv(M, 64) * cdiv(N, 64) >= 32 && !transA && K >= 32 && K % 32 == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
                    (transB || N % 4 == 0) && aligned16(A) && aligned16(B) && bias_kind != SOFIE_BIAS_FULL &&
                    (size_t)128 * lda * 4 < (1u << 31) && (size_t)(transB ? 128 : K) * ldb * 4 < (1u << 31) &&
                    (size_t)128 * ldy * 4 < (1u << 31) && (size_t)cdiv(M, tile) * cdiv(N, tile) < (1u << 30);
   // a few rows of A on a B of some size: a pass over B (k_gemm_f32_skinny); needs whole 16-byte chunks per lane. With 33 to
   // 64 rows and thousands of column tiles the 64 x 64 tiles below fill the device and reuse B from LDS.
   // ... and more than 32 rows on 16 M elements of B are faster on tiles with K in slices: 64 x 4096 x 4096 27 against 39 us.
   // (Both this rule and the one for `dma` on few tiles are wider than the times say, us here / in launch_general: 64 x 512 x 512
   // 14.2 / 5.3, 32 x 4096 x 4096 26.2 / 19.0, 1 x 1024 x 8192 10.7 / 12.2; 256 x 512 x 512 11.4 / 5.9, 512 x 1024 x 1024 19.4 /
   // 14.0. test_gemm_f32_few_rows and test_gemm_f32_few_tiles_long_k_in_slices name the kernels that run inside them.)
   const bool skinny = (M <= 32 || (M <= 64 && N < 8192 && (size_t)N * K < ((size_t)1 << 24))) && !transA && K >= 64 && K % 4 == 0 && (size_t)N * K >= 64 * 1024 && lda % 4 == 0 && ldb % 4 == 0 &&
                       (transB || N % 4 == 0) && aligned16(A) && aligned16(B) &&
                       (size_t)M * lda * 4 < (1u << 31) && (size_t)(transB ? N : K) * ldb * 4 < (1u << 31) &&
                       (size_t)M * ldy < (1u << 31);
   if (skinny) return launch_skinny(ctx, g);
   // tiles for less than half of the compute units and a K of 16 steps or more: K in slices (of at least 8 steps) so that about two
   // workgroups per compute unit exist; the slices' sums are added by the pass of the few-rows kernel
   // (128 x 1024 x 4096: 18.5 against 76.9 us; with a tile for every compute unit slices gain and lose: -6 % .. +14 %)
   const int tiles = dma ? cdiv(M, tile) * cdiv(N, tile) : 0, steps = K / 32;
   const bool sliced = small && tiles * 2 <= ctx->num_cus && steps >= 16;
   // k_gemm_f32_split instead of whole tiles of 24 us and more (by kTileCosts; below that it gains little, and test_gemm_f32_large
   // names the kernels): us 2048^3 137 / 124, 4096 x 4096 x 3000 700 / 636; 1024^3 here, 22
   bool split = false;
   if (dma && !sliced) {
      const int per_cu = cdiv(tiles, ctx->num_cus);
      const TileCost &t = small ? kTileCosts[3] : kTileCosts[5];
      const float us = 2.0f + (per_cu == 1 ? t.alone : (float)per_cu * t.among) * steps;
      split = us >= 24.0f && (gemm_f32_split_choice(ctx, g, 1, true).us < us || gemm_f32_shared_choice(ctx, g, 1).us < us);
   }
   if (dma && !split) {
      constexpr auto kern_nk2 = k_gemm_f32_dma<false, 2>, kern_kn2 = k_gemm_f32_dma<true, 2>;
      constexpr auto kern_nk1 = k_gemm_f32_dma<false, 1>, kern_kn1 = k_gemm_f32_dma<true, 1>;
      SOFIE_LARGE_LDS(kern_nk2);
      SOFIE_LARGE_LDS(kern_kn2);
      SOFIE_LARGE_LDS(kern_nk1);
      SOFIE_LARGE_LDS(kern_kn1);
      const auto kern = small ? (transB ? kern_nk1 : kern_kn1) : (transB ? kern_nk2 : kern_kn2);
      int splits = 1;
      if (sliced) {
         splits = 2 * ctx->num_cus / tiles;
         if (splits > steps / 8) splits = steps / 8;
         if (splits > 16) splits = 16;
         splits = cdiv(steps, cdiv(steps, splits));
      }
      if (splits > 1) {
         void *ws = nullptr;
         if (int rc = workspace(ctx, (size_t)splits * M * N * sizeof(float), &ws)) return rc;
         g.partial = static_cast<float *>(ws);
      }
      hipLaunchKernelGGL(kern, dim3(tiles, splits), dim3(256), 2 * (tile + tile) * 32 * 4, ctx->stream, g);
      if (int rc = check_launch(ctx, small ? "k_gemm_f32_dma64" : "k_gemm_f32_dma")) return rc;
      if (splits == 1) return SOFIE_HIP_OK;
      return launch_finish(ctx, g, splits);
   }
   // (a bias given for every output element keeps to one launch)
   return launch_general(ctx, g, 1, bias_kind == SOFIE_BIAS_FULL);
}

extern "C" int sofie_hip_gemm_f32_stacked(sofie_hip_ctx *ctx, int transA, int transB, int M, int N, int K, float alpha,
                                          const float *A, int lda, const float *B, int ldb, float *Y, int ldy, int n_lead,
                                          const int *lead, const long long *stride_a, const long long *stride_b, int act)
{
   if (!ctx) return SOFIE_HIP_EINVAL;
   SOFIE_REQUIRE(ctx, M >= 0 && N >= 0 && K >= 0, "negative dimension");
   SOFIE_REQUIRE(ctx, n_lead >= 1 && n_lead <= SOFIE_GEMM_MAX_LEAD && lead && stride_a && stride_b, "bad leading dimensions");
   SOFIE_REQUIRE(ctx, act == SOFIE_ACT_NONE || act == SOFIE_ACT_RELU, "unknown activation");
   long long stack = 1;
   for (int d = 0; d < n_lead; ++d) {
      SOFIE_REQUIRE(ctx, lead[d] >= 0 && stride_a[d] >= 0 && stride_b[d] >= 0, "negative extent or stride");
      stack *= lead[d];
      SOFIE_REQUIRE(ctx, stack < (1ll << 31), "too many stacked products");
   }
   if (M == 0 || N == 0 || stack == 0) return SOFIE_HIP_OK;
   SOFIE_REQUIRE(ctx, Y && (K == 0 || (A && B)), "null operand");
   SOFIE_REQUIRE(ctx, lda >= (transA ? M : K) && ldb >= (transB ? K : N) && ldy >= N, "leading dimension too small");
   GemmF32Args g{};
   g.A = A; g.B = B; g.bias = nullptr; g.Y = Y;
   g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldb = ldb; g.ldy = ldy;
   g.transA = transA != 0; g.transB = transB != 0;
   g.alpha = alpha; g.beta = 0.0f; g.bias_kind = SOFIE_BIAS_NONE; g.relu = act == SOFIE_ACT_RELU;
   g.n_lead = n_lead;
   for (int d = 0; d < n_lead; ++d) { g.lead[d] = lead[d]; g.sa[d] = stride_a[d]; g.sb[d] = stride_b[d]; }
   g.stride_y = (long long)M * ldy;
   // the grid's third dimension holds at most 65535 products per launch
   for (long long z0 = 0; z0 < stack; z0 += 65535) {
      const unsigned nz = (unsigned)((stack - z0) < 65535 ? (stack - z0) : 65535);
      g.z0 = (int)z0;
      if (int rc = launch_general(ctx, g, nz, true)) return rc;
   }
   return SOFIE_HIP_OK;
}

// ------------------------------------------------------------------------------------------------------------
// A chain of small fully connected layers in one launch: y = act_L(... act_1(x W_1 + b_1) ... W_L + b_L).
// A workgroup carries 16 RT rows through every layer with the activations in LDS, on v_mfma_f32_16x16x4_f32. The weights
// (W_l [K_l, N_l], row-major) go straight from the L2 into the instruction's operand registers, 4 bytes per lane of any
// dword: a piece is 64 rows of k x 16 columns, 16 loads. A wavefront's pieces form one list over all column tiles, parts of K and
// layers, and the loads of the next piece are always under way while one is multiplied: the first weights (and biases) of a layer
// arrive under the layer before it. Against one thread per output and 1, 4 or 8 rows per workgroup (us): 64-128-64-8 on 256 rows
// 7.5 -> 6.6, on 16384 27.4 -> 12.5; 20-32-32-1 on 4096 15.5 -> 5.3; 100-487-13 on 8192 34.8 -> 16.7. The arguments of a layer in one scalar
// load, those of the first four layers fetched at the start, x ahead of the weights: 64-128-64-8 on 256 rows 6.6 -> 5.9, 60 random
// chains (k_mlp_f32_row's, too) 1.065 times shorter in the mean, none longer (with units dealt on from layer to layer, so that idle
// wavefronts ask for the next layer's weights, 6.05). What bounds it: launch and
// memory latency for a small network on a few rows; a compute unit's share of the L2 (43 B/ns measured, every workgroup reads all
// weights) up to 16 rows for each of them; the matrix instructions above.
// A layer with fewer column tiles than the workgroup has wavefronts deals the pieces of K to parts, added in LDS in order.
namespace {

struct MlpLayer {      // 32 bytes: one scalar load
   const float *W, *bias;
   int K, N, relu;
   int psh;      // k_mlp_f32: the pieces of K are dealt to 1 << psh parts
};

struct MlpArgs {
   const float *x;
   float *y;
   int n_layers, M, ldx, ldy;
   int ld[2];   // floats per row of the two activation buffers: the inputs of even and of odd layers
   int maxd;    // k_mlp_f32_row: the widest layer
   alignas(64) MlpLayer layer[SOFIE_MLP_MAX_LAYERS];
};

template <int RT, int NW>
__global__ void __launch_bounds__(NW * 64) k_mlp_f32(MlpArgs a)
{
   constexpr int ROWS = 16 * RT;
   // sums per output: shorter chains of rounded additions, and matrix instructions that do not wait for each other
   constexpr int CH = RT == 4 ? 2 : 4;
   extern __shared__ __align__(16) float s_mlp[];
   float *const buf[2] = {s_mlp, s_mlp + ROWS * a.ld[0]};
   float *const part = s_mlp + ROWS * (a.ld[0] + a.ld[1]);     // [wavefront][RT][lane][4] sums of parts of K
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int c = lane & 15, kg = lane >> 4;
   const int row0 = blockIdx.x * ROWS;
   ask_for_arguments<3 * 64>();      // up to the fourth layer

   // the next piece whose weights are requested: layer, unit (column tile and part), piece of K; and what its layer's pieces share
   int fl = -1, fu = 0, fp = 0, fK = 0, fN = 0, fsh = 0, funits = 0;
   __amdgpu_buffer_rsrc_t fw, fb;
   auto settle = [&] {       // onto the first piece of this wavefront at or behind unit fu
      while (fu >= funits) {
         if (++fl >= a.n_layers) return;
         const MlpLayer f = a.layer[fl];
         fK = f.K;
         fN = f.N;
         fsh = f.psh;
         funits = ((fN + 15) >> 4) << fsh;
         fu = wave;
         // rows behind K lie outside the descriptor and arrive as zeros; columns behind N hold other weights and end in
         // columns of the result that are dropped
         fw = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(f.W), 0, fK * fN * 4, 0x00020000);
         fb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(f.bias), 0, f.bias ? fN * 4 : 0, 0x00020000);
      }
      fp = fu & ((1 << fsh) - 1);
   };
   float nw[16], nb = 0.0f;
   auto fetch = [&] {
      if (fl >= a.n_layers) return;
      const int n = (fu >> fsh) * 16 + c, row = fN * 4;
      const int at = (fp * 64 + 4 * kg) * row + n * 4;
#pragma unroll
      for (int s = 0; s < 4; ++s)
         if (fp * 64 + s * 16 < fK) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
               nw[4 * s + e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(fw, at + (16 * s + e) * row, 0, 0));
         }
      nb = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(fb, n * 4, 0, 0));
      fp += 1 << fsh;
      if (fp * 64 >= fK) {
         fu += NW;
         settle();
      }
   };
   // the rows of x, with zeros up to a whole 16 of K and for rows behind M; the first 64 columns are requested ahead of the weights
   const int K0 = a.layer[0].K;
   float v[ROWS / NW];
   auto request_x = [&](int k) {
#pragma unroll
      for (int i = 0; i < ROWS / NW; ++i) {
         const int row = row0 + i * NW + wave;
         v[i] = row < a.M && k < K0 ? a.x[(size_t)row * a.ldx + k] : 0.0f;
      }
   };
   request_x(lane);
   settle();
   fetch();
   for (int k = lane, KP = (K0 + 15) & ~15; k < KP; k += 64) {
      if (k >= 64) request_x(k);
#pragma unroll
      for (int i = 0; i < ROWS / NW; ++i) buf[0][(i * NW + wave) * a.ld[0] + k] = v[i];
   }
   __syncthreads();

   for (int l = 0; l < a.n_layers; ++l) {
      const MlpLayer f = a.layer[l];
      const int K = f.K, N = f.N, ldi = a.ld[l & 1], ldo = a.ld[(l + 1) & 1];
      const float *in = l & 1 ? buf[1] : buf[0];
      float *out = l & 1 ? buf[0] : buf[1];
      const bool last = l + 1 == a.n_layers, relu = f.relu;
      const int sh = f.psh, parts = 1 << sh, tiles = (N + 15) >> 4, pieces = (K + 63) >> 6;
      // columns behind N become the zeros up to a whole 16 of the next layer's K
      auto finish = [&](int r, int n, float v) {
         if (relu) v = fmaxf(v, 0.0f);
         if (!last) out[r * ldo + n] = n < N ? v : 0.0f;
         else if (n < N && row0 + r < a.M) a.y[(size_t)(row0 + r) * a.ldy + n] = v;
      };
      for (int u = wave; u < tiles << sh; u += NW) {
         const int t = u >> sh, p = u & (parts - 1);
         v4f acc[RT][CH];
#pragma unroll
         for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int h = 0; h < CH; ++h) acc[i][h] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
         float bias = 0.0f;
         for (int q = p; q < pieces; q += parts) {
            float w[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) w[e] = nw[e];
            bias = nb;
            fetch();
            const float *ap = in + c * ldi + q * 64 + 4 * kg;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
               if (q * 64 + s * 16 >= K) break;
#pragma unroll
               for (int i = 0; i < RT; ++i) {
                  const v4f f = *reinterpret_cast<const v4f *>(ap + i * 16 * ldi + s * 16);
#pragma unroll
                  for (int e = 0; e < 4; ++e) acc[i][e % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[e], w[4 * s + e], acc[i][e % CH], 0, 0, 0);
               }
            }
         }
         // a lane has rows 4 kg .. 4 kg + 3 of column c
#pragma unroll
         for (int i = 0; i < RT; ++i) {
            v4f sum = acc[i][0] + acc[i][1];
            if constexpr (CH == 4) sum += acc[i][2] + acc[i][3];
            if (p == 0) sum += bias;
            if (parts > 1) *reinterpret_cast<v4f *>(part + ((u * RT + i) * 64 + lane) * 4) = sum;
#pragma unroll
            for (int e = 0; e < 4; ++e)
               if (parts == 1) finish(i * 16 + kg * 4 + e, t * 16 + c, sum[e]);
         }
      }
      if (parts > 1) {
         __syncthreads();
         for (int idx = tid; idx < tiles * RT * 256; idx += NW * 64) {
            const int t = idx / (RT * 256), o = idx - t * (RT * 256), ln = (o >> 2) & 63, n = t * 16 + (ln & 15);
            float v = part[t * parts * (RT * 256) + o];
            for (int p = 1; p < parts; ++p) v += part[(t * parts + p) * (RT * 256) + o];
            finish((o >> 8) * 16 + (ln >> 4) * 4 + (o & 3), n, v);
         }
      }
      __syncthreads();
   }
}

// One row per workgroup and one output per thread, plain fused multiply-adds: a layer of fewer than 256 outputs is cut into parts of
// K whose sums meet in LDS. For up to two rows per compute unit, where it is the shorter chain of waits (us, against k_mlp_f32):
// 144-128-41 on 256 rows 6.1 / 7.2, 147-112-128-32-95-23 10.8 / 12.2, 8-500-9 6.1 / 6.6; not with a layer of 8 outputs or fewer
// (32 parts and more, added one after the other): 64-128-64-8 7.5 / 5.9, 20-32-32-1 16.0 / 5.3.
__global__ void __launch_bounds__(256) k_mlp_f32_row(MlpArgs a)
{
   constexpr int R = 1;
   extern __shared__ __align__(16) float s_mlp[];
   float *buf_in = s_mlp, *buf_out = s_mlp + R * a.maxd;     // activations of the rows, [R][maxd] each
   float *part = s_mlp + 2 * R * a.maxd;                     // [256][R] partial sums
   const int tid = threadIdx.x;
   const int row0 = blockIdx.x * R;
   {
      const int K0 = a.layer[0].K;
      for (int idx = tid; idx < R * K0; idx += 256) {
         const int r = idx / K0, k = idx - r * K0;
         buf_in[r * a.maxd + k] = row0 + r < a.M ? a.x[(size_t)(row0 + r) * a.ldx + k] : 0.0f;
      }
   }
   __syncthreads();
   for (int l = 0; l < a.n_layers; ++l) {
      const MlpLayer f = a.layer[l];
      const int K = f.K, N = f.N;
      const float *__restrict__ W = f.W;
      const bool last = l + 1 == a.n_layers;
      // columns per pass (a power of two, at most 256) and the parts K is cut into
      int n2 = 1;
      while (n2 < N && n2 < 256) n2 <<= 1;
      const int parts = 256 / n2;
      const int kc = (K + parts - 1) / parts;
      const int oc = tid & (n2 - 1), pt = tid / n2;
      const int k0 = pt * kc, k1 = k0 + kc < K ? k0 + kc : K;
      for (int o0 = 0; o0 < N; o0 += n2) {
         const int o = o0 + oc;
         float acc[R];
#pragma unroll
         for (int r = 0; r < R; ++r) acc[r] = 0.0f;
         if (o < N) {
            const float *w = W + (size_t)k0 * N + o;
#pragma unroll 8
            for (int k = k0; k < k1; ++k) {
               const float wv = *w;
               w += N;
#pragma unroll
               for (int r = 0; r < R; ++r) acc[r] = fmaf(buf_in[r * a.maxd + k], wv, acc[r]);
            }
         }
         auto finish = [&](int r, int oo, float v) {
            if (f.bias) v += f.bias[oo];
            if (f.relu) v = fmaxf(v, 0.0f);
            if (last) {
               if (row0 + r < a.M) a.y[(size_t)(row0 + r) * a.ldy + oo] = v;
            } else {
               buf_out[r * a.maxd + oo] = v;
            }
         };
         if (parts == 1) {
            // 256 columns per pass: every thread holds the complete sums of its column
            if (o < N) {
#pragma unroll
               for (int r = 0; r < R; ++r) finish(r, o, acc[r]);
            }
         } else {
#pragma unroll
            for (int r = 0; r < R; ++r) part[tid * R + r] = acc[r];
            __syncthreads();
            // the parts of an output are added in order by one thread per (row, output)
            for (int idx = tid; idx < R * n2; idx += 256) {
               const int r = idx / n2, c = idx - r * n2;
               if (o0 + c >= N) continue;
               float v = 0.0f;
               for (int p = 0; p < parts; ++p) v += part[(p * n2 + c) * R + r];
               finish(r, o0 + c, v);
            }
         }
         if (parts > 1) __syncthreads();   // the partial sums are read before the next pass overwrites them
      }
      __syncthreads();
      float *t = buf_in; buf_in = buf_out; buf_out = t;
   }
}

template <int RT, int NW>
int launch_mlp(sofie_hip_ctx *ctx, MlpArgs &a, size_t lds)
{
   SOFIE_LARGE_LDS((k_mlp_f32<RT, NW>));
   for (int l = 0; l < a.n_layers; ++l) {
      MlpLayer &f = a.layer[l];
      const int tiles = cdiv(f.N, 16), pieces = cdiv(f.K, 64);
      for (f.psh = 0; (2 * tiles << f.psh) <= NW && (2 << f.psh) <= pieces;) ++f.psh;
   }
   // a launch holds fewer than 2^32 threads: 67 million rows at 16 per workgroup of 1024
   const int M = a.M, most = (1 << 21) * 16 * RT;
   for (int row = 0;; row += most) {
      a.M = M - row < most ? M - row : most;
      hipLaunchKernelGGL((k_mlp_f32<RT, NW>), dim3((unsigned)cdiv(a.M, 16 * RT)), dim3(NW * 64), lds, ctx->stream, a);
      if (int rc = check_launch(ctx, "k_mlp_f32")) return rc;
      if (M - row <= most) return SOFIE_HIP_OK;
      a.x += (size_t)most * a.ldx;
      a.y += (size_t)most * a.ldy;
   }
}

// A layer as a product of its own (lda and ldy: of x and y for the first and the last, else of the scratch buffer).
GemmF32Args mlp_layer(const MlpArgs &a, int l, const float *in, int lda, float *out, int ldy)
{
   const MlpLayer &f = a.layer[l];
   GemmF32Args g{};
   g.A = in; g.B = f.W; g.bias = f.bias; g.Y = out;
   g.M = a.M; g.N = f.N; g.K = f.K;
   g.lda = lda; g.ldb = g.N; g.ldy = ldy;
   g.alpha = 1.0f; g.beta = f.bias ? 1.0f : 0.0f;
   g.bias_kind = f.bias ? SOFIE_BIAS_ROW : SOFIE_BIAS_NONE;
   g.relu = f.relu;
   return g;
}

}  // namespace

extern "C" int sofie_hip_mlp_f32(sofie_hip_ctx *ctx, int n_layers, const int *dims, const float *const *W,
                                 const float *const *bias, const int *act, const float *x, int ldx, float *y, int ldy,
                                 int M)
{
   if (!ctx) return SOFIE_HIP_EINVAL;
   SOFIE_REQUIRE(ctx, n_layers >= 1 && n_layers <= SOFIE_MLP_MAX_LAYERS && dims && W && act, "bad layer list");
   SOFIE_REQUIRE(ctx, M >= 0, "negative dimension");
   MlpArgs a{};
   for (int l = 0; l <= n_layers; ++l) {
      SOFIE_REQUIRE(ctx, dims[l] >= 1 && dims[l] <= SOFIE_MLP_MAX_WIDTH, "layer width out of range");
      if (l < n_layers) a.layer[l].K = dims[l];
      if (l > 0) a.layer[l - 1].N = dims[l];
   }
   for (int l = 0; l < n_layers; ++l) {
      SOFIE_REQUIRE(ctx, W[l], "null weight matrix");
      SOFIE_REQUIRE(ctx, act[l] == SOFIE_ACT_NONE || act[l] == SOFIE_ACT_RELU, "unknown activation");
      a.layer[l].W = W[l];
      a.layer[l].bias = bias ? bias[l] : nullptr;
      a.layer[l].relu = act[l] == SOFIE_ACT_RELU;
   }
   if (M == 0) return SOFIE_HIP_OK;
   SOFIE_REQUIRE(ctx, x && y, "null operand");
   SOFIE_REQUIRE(ctx, ldx >= dims[0] && ldy >= dims[n_layers], "leading dimension too small");
   a.x = x; a.y = y; a.n_layers = n_layers; a.M = M; a.ldx = ldx; a.ldy = ldy;
   // a row of a buffer: the widest layer it holds, up to a whole 16, and 4 floats that keep neighbouring rows on other banks
   for (int l = 0; l < n_layers; ++l) {
      const int w = ((dims[l] + 15) & ~15) + 4;
      if (w > a.ld[l & 1]) a.ld[l & 1] = w;
   }
   auto lds = [&](int rt, int waves) { return (size_t)(16 * rt * (a.ld[0] + a.ld[1]) + waves * rt * 256) * sizeof(float); };
   // 16 rows per workgroup while that is at most one workgroup per compute unit; more rows share a pass over the weights above
   // it, as far as the activations fit (16 rows of the widest layers take 148 KB)
   const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
   const int rt = M > 64 * cus && lds(4, 8) <= (size_t)kMaxDynamicLds ? 4 : M > 16 * cus && lds(2, 8) <= (size_t)kMaxDynamicLds ? 2 : 1;
   // In one launch every workgroup takes in all weights, 43 bytes per ns and compute unit, which a launch per layer (2.8 us each)
   // shares out: the shorter estimate, and a single layer is a product in any case. One launch against a launch per layer:
   // 64-128-64-8 on 256 rows 5.9 / 13.4 us, 256-256-256-16 on 512 rows 18.5 / 12.8, 1024-1024-1024 on 256 rows 199 / 22.5.
   // (k_mlp_f32_row: the weights as often as a compute unit has rows; 8-16-768 on 8 rows 6.0 us, 6.9 in two launches.)
   const int per_cu = cdiv(cdiv(M, 16 * rt), cus);
   int narrowest = dims[1];
   float one = 3.0f + n_layers, each = 0.0f, row = one;
   for (int l = 0; l <= n_layers; ++l) {
      if (dims[l] > a.maxd) a.maxd = dims[l];
      if (l > 0 && dims[l] < narrowest) narrowest = dims[l];
   }
   const bool by_rows = M <= 2 * cus && narrowest > 8;
   for (int l = 0; l < n_layers; ++l) {
      const float weights = (float)((dims[l] + 63) & ~63) * (float)((dims[l + 1] + 15) & ~15);
      const float reads = weights * 4.0f / 43e3f, mfma = weights * 32.0f * rt / 550e3f;
      one += per_cu * (reads > mfma ? reads : mfma);
      row += cdiv(M, cus) * 4.0f * dims[l] * dims[l + 1] / 43e3f;
      each += 2.8f + general_choice(ctx, mlp_layer(a, l, x, dims[l], y, dims[l + 1]), 1, true).us;
   }
   int widest = 0;
   for (int l = 1; l < n_layers; ++l)
      if (dims[l] > widest) widest = dims[l];
   // (memory between the layers: without it, as while a graph is recorded on a context that has none, one launch does. One
   // layer written over its own input stays with the kernels that take in a workgroup's rows before they write them.)
   const size_t floats = (size_t)M * widest;
   const bool in_place = n_layers == 1 && x < y + (size_t)(M - 1) * ldy + dims[1] && y < x + (size_t)(M - 1) * ldx + dims[0];
   if (((n_layers == 1 && !in_place) || (n_layers > 1 && each < (by_rows && row < one ? row : one))) && ldx < (1 << 22) && floats < ((size_t)1 << 28)) {
      float *const ws = n_layers == 1 ? nullptr : static_cast<float *>(workspace_if_room(ctx, 2 * floats * sizeof(float)));
      if (n_layers == 1 || ws) {
         const float *in = x;
         int lda = ldx;
         for (int l = 0; l < n_layers; ++l) {
            const bool last = l + 1 == n_layers;
            float *out = last ? y : ws + (l & 1) * floats;
            GemmF32Args g = mlp_layer(a, l, in, lda, out, last ? ldy : dims[l + 1]);
            if (int rc = launch_general(ctx, g, 1, true)) return rc;
            in = out;
            lda = dims[l + 1];
         }
         return SOFIE_HIP_OK;
      }
   }
   if (by_rows) {
      hipLaunchKernelGGL(k_mlp_f32_row, dim3((unsigned)M), dim3(256), (2 * a.maxd + 256) * sizeof(float), ctx->stream, a);
      return check_launch(ctx, "k_mlp_f32_row");
   }
   if (rt == 4) return launch_mlp<4, 8>(ctx, a, lds(4, 8));
   if (rt == 2) return launch_mlp<2, 8>(ctx, a, lds(2, 8));
   return launch_mlp<1, 16>(ctx, a, lds(1, 16));
}
