// One operand tile of k_gemm_f32 (gemm_f32.hip): which bytes of the matrix a lane asks for in a K-step, and where in the LDS they
// go. The index arithmetic alone, on rsrc_t, make_rsrc, dma16 and dma4 of gemm_tile.h (or of a host program that checks the
// addresses).
#pragma once

namespace sofie {

template <bool KM, int ROWS>
struct F32Operand {
   static constexpr int BK = 32;
   static constexpr int NRQ = ROWS / 32;                                             // requests per stage
   static constexpr int NV = KM ? (ROWS == 128 ? 2 : ROWS == 96 ? 3 : 1) : 1;        // different lane offsets among them
   static constexpr int KPR = 1024 / ROWS;                                           // KM: rows of k per request (but for 96 columns)
   static constexpr unsigned OUTSIDE = 0x80000000u;
   const float *base;
   rsrc_t rs;                      // rows along K: the tile's rows
   unsigned voff[NV];
   int kofs[NV];                   // first k of the lane's 16 bytes inside the stage (KM: of the request)
   unsigned ld4;
   int ld, K, rows, first, tid;
   bool straddles;                 // the last step has pieces that are inside in part
   unsigned row_offset[KM ? 1 : NRQ];      // rows along K: uniform offsets of the requests' rows

   __device__ __forceinline__ void init(const float *base_, int ld_, int first_, int count, int K_, int tid_)
   {
      ld = ld_;
      ld4 = (unsigned)ld_ * 4u;
      K = K_;
      first = first_;
      tid = tid_;
      rows = count - first < ROWS ? count - first : ROWS;
      if constexpr (KM) {
         base = base_ + first;
         straddles = (rows & 3) != 0;
#pragma unroll
         for (int v = 0; v < NV; ++v) {
            const int idx = v * 256 + tid, k = idx / (ROWS / 4), pos = idx % (ROWS / 4) * 4;
            const int col = (pos + ROWS - 16 * ((k >> 2) & 3) % ROWS) % ROWS;
            kofs[v] = NV == 2 ? k - v * KPR : k;
            voff[v] = col < rows ? (unsigned)kofs[v] * ld4 + (unsigned)col * 4u : OUTSIDE;
         }
      } else {
         base = base_ + (size_t)first * ld;
         straddles = (K & 3) != 0;
         rs = make_rsrc(base, (unsigned)rows * ld4);
         const int row = tid >> 3;
         kofs[0] = ((tid & 7) ^ ((row >> 1) & 7)) * 4;
         voff[0] = (unsigned)row * ld4 + (unsigned)kofs[0] * 4u;
#pragma unroll
         for (int u = 0; u < NRQ; ++u) row_offset[u] = u * 32 < rows ? (unsigned)u * 32u * ld4 : 0u;
      }
   }
   // Steps that may be requested without checks (WHOLE): all of their k exist, and no piece of theirs reaches behind the
   // operand's last element, which with rows along M or N that are no whole fours the last step's pieces would do.
   __device__ __forceinline__ int whole_steps() const { return (KM && straddles ? K - 1 : K) / BK; }
   // The cells of K-step kt into LDS byte address dst. WHOLE: kt < whole_steps() (a wavefront has its SIMD to itself here, so
   // every instruction of the loop is time: no checks). A uniform offset never exceeds the descriptor's range
   // (requests of rows that do not exist ask for the tile's first rows, whose results are not stored).
   template <bool WHOLE>
   __device__ __forceinline__ void request(int kt, unsigned dst, int wave) const
   {
      const int k0 = kt * BK, left = WHOLE ? BK : K - k0 < BK ? K - k0 : BK;
      if constexpr (KM) {
         // a descriptor per step: its rows of k (any number of steps, a matrix of any size)
         const bool last = !WHOLE && k0 + BK >= K;
         const rsrc_t step = make_rsrc(base + (left > 0 ? (size_t)k0 * ld : 0),
                                       left <= 0 ? 0u : last ? (unsigned)(left - 1) * ld4 + (unsigned)rows * 4u : BK * ld4);
         if (!WHOLE && straddles && last && left > 0) {
            for (int u = 0; u < ROWS / 8; ++u) {
               const int idx = u * 256 + tid, k = idx / ROWS, pos = idx % ROWS;
               const int col = (pos + ROWS - 16 * ((k >> 2) & 3) % ROWS) % ROWS;
               dma4(step, dst + u * 1024 + wave * 256, (int)(col < rows && k < left ? (unsigned)k * ld4 + (unsigned)col * 4u : OUTSIDE), 0);
            }
            return;
         }
#pragma unroll
         for (int u = 0; u < NRQ; ++u) {
            const int k = NV == 3 ? 0 : u * KPR;
            const unsigned v = WHOLE || k + kofs[u % NV] < left ? voff[u % NV] : OUTSIDE;
            dma16(step, dst + u * 4096 + wave * 1024, (int)v, (int)(WHOLE || k < left ? (unsigned)k * ld4 : 0u));
         }
      } else {
         const unsigned k4 = left > 0 ? (unsigned)k0 * 4u : 0u;
         if (!WHOLE && straddles && left < BK && left > 0) {
            for (int u = 0; u < ROWS / 8; ++u) {
               const int row = u * 8 + (tid >> 5), pos = tid & 31;
               const int k = (((pos >> 2) ^ ((row >> 1) & 7)) << 2) + (pos & 3);
               dma4(rs, dst + u * 1024 + wave * 256, (int)(row < rows && k < left ? (unsigned)row * ld4 + (unsigned)k * 4u : OUTSIDE), (int)k4);
            }
            return;
         }
         const unsigned v = WHOLE || kofs[0] < left ? voff[0] : OUTSIDE;
#pragma unroll
         for (int u = 0; u < NRQ; ++u) dma16(rs, dst + u * 4096 + wave * 1024, (int)v, (int)(row_offset[u] + k4));
      }
   }
};

}  // namespace sofie
