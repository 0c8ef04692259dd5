// fp32 products on the bf16 matrix instructions with every operand as three bf16 numbers (split_bf16.h): k_gemm_f32_split.
//
// A workgroup owns 16 MI rows x 64 columns; its eight wavefronts take the chunks of 32 k in turn, each for the whole tile (MI x 4 tiles
// of 16 x 16), and their sums meet in LDS in a fixed order. An operand of the tile is split once, and wavefronts share nothing on the
// way: each has a buffer of its own in LDS for a chunk of both operands, memory -> LDS without registers (16 bytes per lane, which
// takes any address on a dword), no barrier in the loop. The next chunk is requested as soon as the registers have the one before.
//   * an operand with rows along K lies in rows of 32 k; lane group kg takes k = 4 kg .. + 3 and 16 + 4 kg .. + 3 of its row;
//   * one with rows along M or N lies in 32 rows of 64 columns; a lane takes 4 columns of rows 4 kg + u and 16 + 4 kg + u. Element e of
//     the four belongs to tile e of four: a tile is every fourth column, and nothing is transposed.
// Both give lane group kg the same eight k of a chunk, in the same order.
// Rows and columns behind the matrix are copies of the last ones (of the last four, where four are loaded at once: the same sums,
// stored twice, but not those of the tile before: a wavefront that repeats its sums, below, has other last bits than one that does not).
//
// Bound: vector instructions (eleven for two numbers to split, four a tile to add) beside the matrix instructions, which
// run under them only in part: 1.3 us a chunk of 64 rows and SIMD, 0.64 of it matrix instructions. Relative error against 64 bits 7e-8 to
// 1.2e-7 (k_gemm_f32 3e-7 to 1.2e-6). us against k_gemm_f32 and k_gemm_f32_dma: 1500 x 1001 x 1111 33 -> 29; 2048^3 137 -> 124;
// 4096 x 4096 x 3000 700 -> 636; 172 random products it takes 1.17 times shorter in the median, before the factor that split_bf16.h
// multiplies with (3 to 5 % of these). Operands straight into
// registers were no faster at 2048^3 (119; 35 bytes per ns and compute unit), two buffers for each of four wavefronts neither (125).
#include "gemm_f32.h"
#include "gemm_tile.h"
#include "split_bf16.h"

using namespace sofie;

namespace {

constexpr int WAVES = 8, CH = 32, STEP = WAVES * CH, NJ = 4;

__device__ __forceinline__ void wait_requests() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A chunk of T tiles of 16 rows (KM: columns) of one operand, memory -> LDS -> registers. 2048 bytes of LDS a tile.
template <bool KM, int T>
struct SplitOperand {
   static constexpr unsigned OUTSIDE = 0x80000000u;      // no descriptor reaches it
   static constexpr int REQUESTS = 2 * T, BYTES = 2048 * T, NV = KM ? T / 4 : 2 * T;
   const float *base;
   rsrc_t rs;
   unsigned voff[NV], kofs[2];
   unsigned ld4;
   int ld, K, left, width, piece;
   unsigned rd[KM ? 1 : 2];
   __device__ __forceinline__ void init(const float *p, int ld_, int first, int count, int K_, int lane)
   {
      ld = ld_;
      ld4 = (unsigned)ld_ * 4u;
      K = K_;
      const int r16 = lane & 15, kg = lane >> 4, there = count - first;
      if constexpr (KM) {
         // rows of 64 columns; the last four columns may begin in front of the tile: offsets count from one tile earlier
         const int lead = first > 0 ? T * 16 : 0;
         base = p + first - lead;
         width = there + lead;
#pragma unroll
         for (int v = 0; v < NV; ++v) {
            const int c = (v * 16 + r16) * 4;
            voff[v] = (unsigned)kg * ld4 + (unsigned)((c < there - 4 ? c : there - 4) + lead) * 4u;
         }
         rd[0] = (unsigned)(kg * 1024 + r16 * 16);
      } else {
         // rows of eight 16-byte pieces, piece c of row r in slot c ^ ((r >> 1) & 7): the 16 rows a lane group reads with one read
         // per lane fall on 16 slots
         const int rows = there < T * 16 ? there : T * 16;
         base = p + (size_t)first * ld;
         rs = make_rsrc(base, (unsigned)(rows - 1) * ld4 + (unsigned)K * 4u);
         piece = (lane & 7) ^ (lane >> 4);      // of the even requests; the odd ones' rows are eight further: piece ^ 4
#pragma unroll
         for (int v = 0; v < NV; ++v) {
            const int r = v * 8 + (lane >> 3);
            voff[v] = (unsigned)(r < rows ? r : rows - 1) * ld4;
         }
#pragma unroll
         for (int h = 0; h < 2; ++h) rd[h] = (unsigned)(r16 * 128 + (((4 * h + kg) ^ ((r16 >> 1) & 7)) << 4));
      }
   }
   // The chunk at k0 into LDS address dst. Rows behind K arrive as zeros: a descriptor per chunk (a matrix of any size) ends
   // with row K - 1, whose successor's columns lie behind its last one. Four k along a row are moved down to end with K, or outside.
   __device__ __forceinline__ void request(int k0, unsigned dst)
   {
      if constexpr (KM) {
         const int rows = K - k0 < CH ? K - k0 : CH;
         rs = make_rsrc(base + (rows > 0 ? (size_t)k0 * ld : 0), rows > 0 ? (unsigned)(rows - 1) * ld4 + (unsigned)width * 4u : 0u);
#pragma unroll
         for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
               const bool some = 4 * u < rows;      // uniform (an offset of a row that is not there is behind the descriptor's end)
               dma16(rs, dst + v * 8192 + u * 1024, (int)(some ? voff[v] : OUTSIDE), some ? (int)((unsigned)(4 * u) * ld4) : 0);
            }
      } else {
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const int k = k0 + (piece ^ (4 * h)) * 4;
            kofs[h] = k < K - 4 ? (unsigned)k * 4u : k < K ? (unsigned)(K - 4) * 4u : OUTSIDE;
         }
#pragma unroll
         for (int v = 0; v < NV; ++v) dma16(rs, dst + v * 1024, (int)(voff[v] + kofs[v & 1]), 0);
      }
   }
   // lane group kg: k = 4 kg .. + 3 and 16 + 4 kg .. + 3 of the chunk at p
   __device__ __forceinline__ void read(float (&raw)[T][8], const unsigned char *p) const
   {
      if constexpr (KM) {
#pragma unroll
         for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
               const v4f q = *reinterpret_cast<const v4f *>(p + rd[0] + v * 8192 + ((u & 3) + 4 * (u & 4)) * 256);
#pragma unroll
               for (int e = 0; e < 4; ++e) raw[v * 4 + e][u] = q[e];
            }
      } else {
#pragma unroll
         for (int t = 0; t < T; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
               const v4f q = *reinterpret_cast<const v4f *>(p + rd[h] + t * 2048);
#pragma unroll
               for (int e = 0; e < 4; ++e) raw[t][h * 4 + e] = q[e];
            }
      }
   }
   // K that is no whole four: the values of the chunk with the last k at their places, zeros behind them
   __device__ __forceinline__ void trim(float (&raw)[T][8], int k0, int kg) const
   {
      if constexpr (!KM) {
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const int k = k0 + 4 * kg + h * 16, over = k < K ? k - (K - 4) : 0;
#pragma unroll
            for (int t = 0; t < T; ++t) {
               float *r = &raw[t][h * 4];
               if (over > 0) {
                  if (over & 1) { r[0] = r[1]; r[1] = r[2]; r[2] = r[3]; }
                  if (over & 2) { r[0] = r[2]; r[1] = r[3]; }
               }
#pragma unroll
               for (int e = 0; e < 4; ++e) r[e] = k + e < K ? r[e] : 0.0f;
            }
         }
      }
   }
};

template <bool A_KM, bool B_KM, int MI>
__global__ void __launch_bounds__(WAVES * 64, 2) k_gemm_f32_split(GemmF32Args g)
{
   typedef SplitOperand<A_KM, MI> OperandA;
   typedef SplitOperand<B_KM, NJ> OperandB;
   constexpr int V = MI * NJ * 64;                     // quads of output columns of the tile
   constexpr int BUF = OperandA::BYTES + OperandB::BYTES;
   extern __shared__ __align__(16) unsigned char smem_raw[];      // a chunk per wavefront; then the sums
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int kg = lane >> 4;
   if (g.n_lead > 0) select_product(g, (long long)blockIdx.z + g.z0);
   int tm, tn;
   tile_of(blockIdx.x, (g.M + 16 * MI - 1) / (16 * MI), (g.N + 16 * NJ - 1) / (16 * NJ), tm, tn);
   const int m0 = tm * 16 * MI, n0 = tn * 16 * NJ;
   const int chunks = (g.K + CH - 1) / CH;
   int k_begin = 0, k_end = g.K;
   if (gridDim.y > 1) {      // K in slices: raw sums into the slice's plane of the scratch buffer
      const int per = (chunks + (int)gridDim.y - 1) / (int)gridDim.y;
      k_begin = (int)blockIdx.y * per * CH;
      k_end = k_begin + per * CH < g.K ? k_begin + per * CH : g.K;
      g.Y = g.partial + (size_t)blockIdx.y * g.M * g.N;
      g.ldy = g.N;
      g.alpha = 1.0f;
      g.bias_kind = SOFIE_BIAS_NONE;
      g.relu = 0;
   }
   OperandA oa;
   OperandB ob;
   oa.init(g.A, g.lda, m0, g.M, g.K, lane);
   ob.init(g.B, g.ldb, n0, g.N, g.K, lane);
   unsigned char *const mine = smem_raw + wave * BUF;
   const unsigned mine0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw + (unsigned)(wave * BUF);
   auto request = [&](int k) {      // (behind the slice: outside, zeros)
      ob.request(k < k_end ? k : g.K, mine0);
      oa.request(k < k_end ? k : g.K, mine0 + OperandB::BYTES);
   };
   float ra[MI][8], rb[NJ][8];
   auto read = [&] {
      wait_requests();
      ob.read(rb, mine);
      oa.read(ra, mine + OperandB::BYTES);
   };
   const bool ragged = (g.K & 3) != 0 && !(A_KM && B_KM);
   int k0 = k_begin + wave * CH;
   request(k0);
   v4f acc[MI][NJ];
#pragma unroll
   for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
   read();
   for (; k0 < k_end; k0 += STEP) {
      wait_lds_reads();      // the chunk is in registers
      request(k0 + STEP);
      if (ragged && k0 + CH > g.K) {
         ob.trim(rb, k0, kg);
         oa.trim(ra, k0, kg);
      }
      v4i b[NJ][3], a[2][3];
#pragma unroll
      for (int j = 0; j < NJ; ++j) split8(rb[j], b[j]);
      split8(ra[0], a[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
         if (i + 1 < MI) split8(ra[i + 1], a[(i + 1) & 1]);
         else read();      // the next chunk, under the last matrix instructions of this one
#pragma unroll
         for (int j = 0; j < NJ; ++j) {
            v4f t = {0.0f, 0.0f, 0.0f, 0.0f};
            constexpr int A[6] = {0, 2, 1, 1, 0, 0}, B[6] = {2, 0, 1, 0, 1, 0};
#pragma unroll
            for (int m = 0; m < 6; ++m) t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, b[j][B[m]]), __builtin_bit_cast(v8b, a[i & 1][A[m]]), t, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = __fadd_rn(acc[i][j][e], t[e]);
         }
         __builtin_amdgcn_sched_barrier(0);
      }
   }
   wait_lds_reads();

   // sums that are not finite: again, with fp32 instructions on the operands as they are (1500 x 1001 x 1111, 29 us: 14 more with one
   // infinity, 28 with one in a hundred)
   v4f none = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
   for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
         for (int e = 0; e < 4; ++e) {
            acc[i][j][e] = __fmul_rn(acc[i][j][e], UNSCALE);
            none[e] = fmaf(acc[i][j][e], 0.0f, none[e]);
         }
   if (__builtin_amdgcn_ballot_w64((none[0] + none[1]) + (none[2] + none[3]) != 0.0f) != 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
         for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      for (k0 = k_begin + wave * CH; k0 < k_end; k0 += STEP) {
         wait_lds_reads();
         request(k0);
         read();
         if (ragged && k0 + CH > g.K) {
            ob.trim(rb, k0, kg);
            oa.trim(ra, k0, kg);
         }
#pragma unroll
         for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
               for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb[j][e], ra[i][e], acc[i][j], 0, 0, 0);
      }
   }

   // ((w0 + w4) + (w1 + w5)) + ...: in a fixed order. A quad is four consecutive columns of a row
   v4f *const red = reinterpret_cast<v4f *>(smem_raw);      // [4][V]
   auto quad = [&](int i, int q) { return B_KM ? v4f{acc[i][0][q], acc[i][1][q], acc[i][2][q], acc[i][3][q]} : acc[i][q]; };
   __syncthreads();
   if (wave >= 4) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
         for (int q = 0; q < NJ; ++q) red[(wave - 4) * V + (i * NJ + q) * 64 + lane] = quad(i, q);
   }
   constexpr int MINE = V / 512;
   int m[MINE], n[MINE];
   v4f bias[MINE];
#pragma unroll
   for (int s = 0; s < MINE; ++s) {
      const int at = s * 512 + tid, ln = at & 63, t = at >> 6, i = t / NJ, q = t % NJ, r = ln & 15, c = B_KM ? 16 * (ln >> 4) + 4 * q : 16 * q + 4 * (ln >> 4);
      m[s] = A_KM ? m0 + (i / 4 * 16 + r) * 4 : m0 + i * 16 + r;
      if constexpr (A_KM) {
         m[s] = m[s] >= g.M ? g.M : (m[s] < g.M - 4 ? m[s] : g.M - 4) + i % 4;
         if (m[s] < m0) m[s] = g.M;      // the tile before's
      }
      n[s] = n0 + c;
      if constexpr (B_KM) n[s] = n[s] >= g.N ? g.N : n[s] < g.N - 4 ? n[s] : g.N - 4;
      bias[s] = bias_row4(g, n[s]);
   }
   __syncthreads();
   if (wave < 4) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
         for (int q = 0; q < NJ; ++q) {
            v4f *const d = red + wave * V + (i * NJ + q) * 64 + lane;
            v4f s = quad(i, q);
            const v4f o = *d;
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = __fadd_rn(s[e], o[e]);
            *d = s;
         }
   }
   __syncthreads();
#pragma unroll
   for (int s = 0; s < MINE; ++s) {
      v4f sum = red[s * 512 + tid];
#pragma unroll
      for (int w = 1; w < 4; ++w)
#pragma unroll
         for (int e = 0; e < 4; ++e) sum[e] = __fadd_rn(sum[e], red[w * V + s * 512 + tid][e]);
      if (m[s] < g.M && n[s] < g.N) store4_from(g, finish4(g, sum, bias[s], m[s], n[s]), m[s], n[s], n0);
   }
}

// ---------------------------------------------------------------------------------------------------------------
// 64 rows of one operand (KM: columns of it), 32 k at a time: what a lane of a wavefront asks for and makes of it. Eight requests of 16 bytes;
// four fragments of 16 rows. The lane's k are 4 kg .. + 3 and 16 + 4 kg .. + 3, as above; KM: fragment e is every fourth column.
template <bool KM>
struct SplitRows {
   static constexpr unsigned OUTSIDE = 0x80000000u;
   const float *base;
   __amdgpu_buffer_rsrc_t rs;
   unsigned voff[KM ? 1 : 4], ld4;
   int ld, K, width, kg4;
   __device__ __forceinline__ void init(const float *p, int ld_, int first, int count, int K_, int lane)
   {
      ld = ld_;
      ld4 = (unsigned)ld_ * 4u;
      K = K_;
      kg4 = 4 * (lane >> 4);
      // (a group that begins behind the matrix: copies of the last rows, sums that nobody stores)
      const int r16 = lane & 15, there = count - first;
      if constexpr (KM) {
         // the last four columns may begin in front of the group: offsets count from the group's start or one group earlier
         const int from = first > 0 ? (there >= 4 ? first - 4 : count - 4) : 0;
         base = p + from;
         width = count - from;
         const int c = first + 4 * r16;
         voff[0] = (unsigned)((c < count - 4 ? c : count - 4) - from) * 4u + (unsigned)kg4 * ld4;
      } else {
         const int from = there > 0 ? first : count - 1, rows = there > 0 ? (there < 64 ? there : 64) : 1;
         base = p + (size_t)from * ld;
         rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, (int)((unsigned)(rows - 1) * ld4 + (unsigned)K * 4u), 0x00020000);
#pragma unroll
         for (int f = 0; f < 4; ++f) voff[f] = (unsigned)(16 * f + r16 < rows ? 16 * f + r16 : rows - 1) * ld4;
      }
   }
   // Rows of k behind K arrive as zeros; four k along a row are moved down to end with K, or outside (trim puts them right).
   __device__ __forceinline__ void request(v4f (&q)[8], int k0)
   {
      if constexpr (KM) {
         const int rows = K - k0 < CH ? K - k0 : CH;
         rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base + (rows > 0 ? (size_t)k0 * ld : 0)), 0, rows > 0 ? (int)((unsigned)(rows - 1) * ld4 + (unsigned)width * 4u) : 0, 0x00020000);
#pragma unroll
         for (int u = 0; u < 8; ++u)
            q[u] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(voff[0] + (unsigned)((u & 3) + 4 * (u & 4)) * ld4), 0, 0));
      } else {
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const int k = k0 + 16 * h + kg4;
            const unsigned at = k < K - 4 ? (unsigned)k * 4u : k < K ? (unsigned)(K - 4) * 4u : OUTSIDE;
#pragma unroll
            for (int f = 0; f < 4; ++f) q[2 * f + h] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(voff[f] + at), 0, 0));
         }
      }
   }
   __device__ __forceinline__ void trim(v4f (&q)[8], int k0) const
   {
      if constexpr (!KM) {
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const int k = k0 + 16 * h + kg4, over = k < K ? k - (K - 4) : 0;
#pragma unroll
            for (int f = 0; f < 4; ++f) {
               v4f &r = q[2 * f + h];
               if (over > 0) {
                  if (over & 1) { r[0] = r[1]; r[1] = r[2]; r[2] = r[3]; }
                  if (over & 2) { r[0] = r[2]; r[1] = r[3]; }
               }
#pragma unroll
               for (int e = 0; e < 4; ++e) r[e] = k + e < K ? r[e] : 0.0f;
            }
         }
      }
   }
   // value e (of eight) of fragment f
   static __device__ __forceinline__ float value(const v4f (&q)[8], int f, int e) { return KM ? q[e][f] : q[2 * f + (e >> 2)][e & 3]; }
};

// Tiles of 128 x 128, four wavefronts of 4 x 4 tiles of 16 x 16: an operand of the tile is split once, for all wavefronts, into fragments in LDS (48 KB a
// chunk of 32 k, read without conflicts as they lie). A wavefront reads the chunk's eight fragments into registers; behind a barrier it multiplies them and
// meanwhile splits the 64 rows it has requested of the next chunk into the same LDS. Two workgroups share a compute unit: one reads while
// the other multiplies.
template <bool A_KM, bool B_KM>
__global__ void __launch_bounds__(256, 2) k_gemm_f32_split_shared(GemmF32Args g)
{
   constexpr int BM = 128, BN = 128;
   extern __shared__ __align__(16) unsigned char smem_raw[];
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int kg = lane >> 4, r16 = lane & 15, wm = wave >> 1, wn = wave & 1;
   if (g.n_lead > 0) select_product(g, (long long)blockIdx.z + g.z0);
   int tm, tn;
   tile_of(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
   const int m0 = tm * BM, n0 = tn * BN;
   const bool ragged = (g.K & 3) != 0;
   v4f acc[4][4];
#pragma unroll
   for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
   // fragments [A 0 .. 7, B 0 .. 7][h, m, l][lane]
   v4i *const mine = reinterpret_cast<v4i *>(smem_raw) + wave * 4 * 192 + lane;
   const v8b *const from_a = reinterpret_cast<const v8b *>(smem_raw) + wm * 4 * 192 + lane, *const from_b = reinterpret_cast<const v8b *>(smem_raw) + (8 + wn * 4) * 192 + lane;
   auto run = [&](auto rows) {
      typedef decltype(rows) Rows;
      v4f q[8];
      v4i part[3];
      float r0, r1;
      // two of a fragment's eight values, a few instructions at a time
      auto pair = [&](int f, int p, int stage) {
         switch (stage) {
         case 0:
            r0 = __fmul_rn(Rows::value(q, f, 2 * p), 65536.0f);
            r1 = __fmul_rn(Rows::value(q, f, 2 * p + 1), 65536.0f);
            part[0][p] = (int)f32x2_to_bf16x2(r0, r1);
            break;
         case 1: case 3:
            r0 -= __uint_as_float((unsigned)part[stage >> 1][p] << 16);
            r1 -= __uint_as_float((unsigned)part[stage >> 1][p] & 0xffff0000u);
            break;
         case 2: case 4: part[stage >> 1][p] = (int)f32x2_to_bf16x2(r0, r1); break;
         }
      };
      auto put = [&](int f) {
#pragma unroll
         for (int t = 0; t < 3; ++t) mine[(f * 3 + t) * 64] = part[t];
      };
      rows.request(q, 0);
      if (ragged && CH > g.K) rows.trim(q, 0);
#pragma unroll
      for (int f = 0; f < 4; ++f) {
#pragma unroll
         for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int t = 0; t < 5; ++t) pair(f, p, t);
         put(f);
      }
      rows.request(q, CH);
      for (int k0 = 0; k0 < g.K; k0 += CH) {
         __syncthreads();
         v8b a[4][3], b[4][3];
#pragma unroll
         for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 3; ++t) {
               a[i][t] = from_a[(i * 3 + t) * 64];
               b[i][t] = from_b[(i * 3 + t) * 64];
            }
         wait_lds_reads();
         __builtin_amdgcn_s_barrier();
         asm volatile("" ::: "memory");
         const int next = k0 + CH;
         if (ragged && next < g.K && next + CH > g.K) rows.trim(q, next);
         __builtin_amdgcn_sched_barrier(0);
         v4f t, before;
#pragma unroll
         for (int n = 0; n < 16; ++n) {
            const int i = n / 4, j = n % 4;
            constexpr int A[6] = {0, 2, 1, 1, 0, 0}, B[6] = {2, 0, 1, 0, 1, 0};
            t = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 6; ++m) {
               t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j][B[m]], a[i][A[m]], t, 0, 0, 0);
               if (m < 5) pair(n / 4, n % 4, m);      // of the next chunk, under this one's matrix instructions
               __builtin_amdgcn_sched_barrier(0);
               if (n > 0 && m >= 1 && m < 5) acc[(n - 1) / 4][(n - 1) % 4][m - 1] = __fadd_rn(acc[(n - 1) / 4][(n - 1) % 4][m - 1], before[m - 1]);
               __builtin_amdgcn_sched_barrier(0);
            }
            before = t;
            if (n % 4 == 3) put(n / 4);
            if (n == 15) rows.request(q, next + CH);
            __builtin_amdgcn_sched_barrier(0);
         }
#pragma unroll
         for (int e = 0; e < 4; ++e) acc[3][3][e] = __fadd_rn(acc[3][3][e], before[e]);
      }
   };
   if (wave < 2) {
      SplitRows<A_KM> rows;
      rows.init(g.A, g.lda, m0 + wave * 64, g.M, g.K, lane);
      run(rows);
   } else {
      SplitRows<B_KM> rows;
      rows.init(g.B, g.ldb, n0 + (wave - 2) * 64, g.N, g.K, lane);
      run(rows);
   }

   // sums that are not finite: again, by this wavefront from the operands as they are (2710x5088x336 84 us, 159 with one infinity, 164 where all sums pass 2^95;
   // 5938x7616x728 568, 653, 1060)
   v4f none = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
   for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
         for (int e = 0; e < 4; ++e) {
            acc[i][j][e] = __fmul_rn(acc[i][j][e], UNSCALE);
            none[e] = fmaf(acc[i][j][e], 0.0f, none[e]);
         }
   const int m1 = m0 + wm * 64, n1 = n0 + wn * 64;
   if (__builtin_amdgcn_ballot_w64((none[0] + none[1]) + (none[2] + none[3]) != 0.0f) != 0) {
      SplitRows<A_KM> ra;
      SplitRows<B_KM> rb;
      ra.init(g.A, g.lda, m1, g.M, g.K, lane);
      rb.init(g.B, g.ldb, n1, g.N, g.K, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
         for (int j = 0; j < 4; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
      for (int k0 = 0; k0 < g.K; k0 += CH) {
         v4f qa[8], qb[8];
         ra.request(qa, k0);
         rb.request(qb, k0);
         if (ragged && k0 + CH > g.K) {
            ra.trim(qa, k0);
            rb.trim(qb, k0);
         }
#pragma unroll
         for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
               for (int j = 0; j < 4; ++j)
                  acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(SplitRows<B_KM>::value(qb, j, e), SplitRows<A_KM>::value(qa, i, e), acc[i][j], 0, 0, 0);
      }
   }
   // a quad is four consecutive columns of a row: with B along N element q of the four tiles. (Rows and columns in front of this wavefront's are another one's)
#pragma unroll
   for (int q = 0; q < 4; ++q) {
      int n = n1 + (B_KM ? 16 * kg + 4 * q : 16 * q + 4 * kg);
      if (n >= g.N) continue;
      if constexpr (B_KM) n = n < g.N - 4 ? n : g.N - 4;
      const v4f bias = bias_row4(g, n);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
         int m = m1 + (A_KM ? 4 * r16 : 16 * i + r16);
         if (m >= g.M) continue;
         if constexpr (A_KM) m = (m < g.M - 4 ? m : g.M - 4) + i;
         if (A_KM && m < m1) continue;
         const v4f v = B_KM ? v4f{acc[i][0][q], acc[i][1][q], acc[i][2][q], acc[i][3][q]} : acc[i][q];
         store4_from(g, finish4(g, v, bias, m, n), m, n, n1);
      }
   }
}

template <bool A_KM, bool B_KM>
int launch_shared(sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz)
{
   constexpr auto kern = k_gemm_f32_split_shared<A_KM, B_KM>;
   hipLaunchKernelGGL(kern, dim3(cdiv(g.M, 128) * cdiv(g.N, 128), 1, nz), dim3(256), 16 * 3072, ctx->stream, g);
   return check_launch(ctx, "k_gemm_f32_split_shared");
}

template <bool A_KM, bool B_KM, int MI>
int launch(sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, int splits)
{
   constexpr auto kern = k_gemm_f32_split<A_KM, B_KM, MI>;
   SOFIE_LARGE_LDS(kern);
   hipLaunchKernelGGL(kern, dim3(cdiv(g.M, 16 * MI) * cdiv(g.N, 16 * NJ), splits, nz), dim3(WAVES * 64), WAVES * (MI + NJ) * 2048, ctx->stream, g);
   return check_launch(ctx, "k_gemm_f32_split");
}

}  // namespace

// By an estimate: 2.5 us around the launch; per workgroup of a compute unit (one at a time) 0.7 + 0.6 MI around its loop and 0.9 + 0.5 MI for
// each chunk of its eight wavefronts; slices as for k_gemm_f32, and 7 % for what the estimates of slices miss. K below a chunk for
// each wavefront stays with the fp32 instructions, as does a bias for every output element (one launch).
SplitChoice sofie::gemm_f32_split_choice(const sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, bool one_launch)
{
   SplitChoice best = {0, 1, 1e30f};
   auto offsets_fit = [](bool km, int ld, int rows) { return (long long)(km ? 32 : rows) * ld * 4 < (1ll << 30); };
   if (g.K < 256 || g.M < 4 || g.N < 4 || g.bias_kind == SOFIE_BIAS_FULL || !offsets_fit(!g.transB, g.ldb, 64)) return best;
   const int cus = ctx->num_cus, chunks = cdiv(g.K, CH);
   for (const int mi : {2, 4, 6}) {
      if ((g.transA && mi != 4) || !offsets_fit(g.transA, g.lda, 16 * mi)) continue;
      const long long tiles = (long long)cdiv(g.M, 16 * mi) * cdiv(g.N, 64);
      if (tiles >= (1ll << 32) / 512) continue;
      for (int s = 1; s <= 32; s = s < 4 ? s + 1 : s * 2) {
         if (s > 1 && (one_launch || chunks / s < WAVES || (size_t)g.M * g.N >= ((size_t)1 << 28))) break;
         const long long per_cu = (tiles * nz * s + cus - 1) / cus;
         const float tile = 0.7f + 0.6f * mi + cdiv(cdiv(chunks, s), WAVES) * (0.9f + 0.5f * mi);
         const float us = s == 1 ? 2.5f + (float)per_cu * tile : 1.07f * (7.5f + (float)per_cu * tile + 8.0f * s * (float)g.M * g.N / 6e6f);
         if (us < best.us) best = {mi, s, us};
      }
   }
   return best;
}

// Tiles of 128 x 128 in one piece, two workgroups to a compute unit: 1.39 us a chunk of each, 8 us around two of them (alone 1.75 and 5). In place of the fp32
// instructions alone, whose sums are further off: the eight wavefronts above have eight shorter sums (993 products 8.2e-8 off 64 bits, here 1.2e-7, 2000 9.6e-8
// and 1.6e-7, fp32 instructions 3e-7 and more), and so they keep what they take, though it is the longer way on large products (4096^3 800
// us, 710 here; 4000 x 4001 x 1002 268, 194). Of 140 random products above 2 GFLOP 12 are its, 11 of them 0.79 times as long in the mean, 616 x 5523 x 1112 71.4 us instead of 68.5. With slices of K this is slow (1500 x 1001 x 1111 44 us: a prologue for seven chunks).
SplitChoice sofie::gemm_f32_shared_choice(const sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz)
{
   const SplitChoice none = {0, 1, 1e30f};
   auto offsets_fit = [](bool km, int ld) { return (long long)(km ? 32 : 64) * ld * 4 < (1ll << 30); };
   if (g.K < 64 || g.M < 4 || g.N < 4 || g.bias_kind == SOFIE_BIAS_FULL || !offsets_fit(!g.transB, g.ldb) || !offsets_fit(g.transA, g.lda)) return none;
   const int cus = ctx->num_cus, chunks = cdiv(g.K, CH);
   const long long tiles = (long long)cdiv(g.M, 128) * cdiv(g.N, 128), per_cu = (tiles * nz + cus - 1) / cus;
   if (tiles >= (1ll << 32) / 256) return none;
   return {8, 1, per_cu == 1 ? 8.0f + 1.75f * chunks : 3.0f + 8.0f * (float)((per_cu + 1) / 2) + 1.39f * (float)per_cu * chunks};
}

int sofie::launch_gemm_f32_split(sofie_hip_ctx *ctx, const GemmF32Args &g, unsigned nz, const SplitChoice &c)
{
   if (c.mi == 8)
      return g.transA ? (g.transB ? launch_shared<true, false>(ctx, g, nz) : launch_shared<true, true>(ctx, g, nz))
                      : (g.transB ? launch_shared<false, false>(ctx, g, nz) : launch_shared<false, true>(ctx, g, nz));
   if (g.transA) return g.transB ? launch<true, false, 4>(ctx, g, nz, c.splits) : launch<true, true, 4>(ctx, g, nz, c.splits);
   switch (c.mi) {
   case 2: return g.transB ? launch<false, false, 2>(ctx, g, nz, c.splits) : launch<false, true, 2>(ctx, g, nz, c.splits);
   case 4: return g.transB ? launch<false, false, 4>(ctx, g, nz, c.splits) : launch<false, true, 4>(ctx, g, nz, c.splits);
   default: return g.transB ? launch<false, false, 6>(ctx, g, nz, c.splits) : launch<false, true, 6>(ctx, g, nz, c.splits);
   }
}
