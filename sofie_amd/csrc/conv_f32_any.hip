// fp32 NCHW convolutions of any channels, kernels, strides, dilations and groups, and the output phases of
// transposed ones, as an implicit GEMM on v_mfma_f32_16x16x4_f32 whose operands go from global memory straight into the
// instruction's registers: k_conv_f32_any.
//
//   Y[oc, pixel] = sum_k W[oc, k] * X[k, pixel],  k = (ic, kh, kw),  pixels of all images in one row
//
// A wavefront owns 16 TI channels x 16 TJ pixels and runs on its own: no barrier and no LDS traffic in the loop but one
// 8-byte read per lane and four k. Tiles of 16 and pixels that run on across images leave little work for padding:
// 187 channels on 18 x 18 planes are 12 tiles of 16 and 324 N / 64 columns.
//   * X: lane (r, kg) asks for k = 4 t + kg of pixel r: the pixel's offset (a register for the whole kernel) plus the
//     tap's offset from a table in LDS, out of the descriptor's range where the tap lies outside the image (a bit per
//     kernel row and column in a register, tested with the tap's two bits). The taps of a channel hit the lines that the
//     first one brought into the L1. The table covers CB channels and is walked once per CB of them (a uniform offset);
//     a second one is for the last block if it is not full.
//   * W: a copy laid out as fragments [oc / 16][k / 16][lane][k / 4 % 4] (k_conv_f32_any_weights, in front of the launch or
//     once per tensor under the constant-weights promise): 16 bytes per lane are the operands of four instructions.
//   * 16 k (a group) are loaded while the 16 before them are multiplied, in the order the compiler finds: loads in one go in
//     front of the matrix instructions, or wavefront priorities around either, cost 3 - 17 %.
// Where tiles are few, KS wavefronts of a workgroup share the k of a tile and add up in LDS, in a fixed order.
//
// Bound: fp32 matrix instructions on a large layer of 48 channels and more (the matrix pipe is busy for 86 % of the kernel's cycles on
// 256x64x56x56 -> 128). On smaller layers and short sums nothing is full: 16x3x224x224 -> 64, 7x7 s2 keeps the matrix pipe busy for
// 53 % and makes 0.55 L1 accesses per cycle and compute unit (18 for a request of 64 values), with a request every 32 cycles; the
// layers of 64 and 128 channels on 20x20 and 10x10 54 % and 0.45. Measured against the kernels for one plane and 64 or 128 channels
// at a time (k_conv2d_f32, k_conv2d_f32_dma; us, constant weights): 16x3x224x224 -> 64, 7x7 s2: 85 -> 53; 256x64x10x10 ->
// 128, 3x3: 52 -> 43; 5x80x20x20 -> 9, 7x7: 370 -> 14; 131x128x96x96 -> 80, 1x1: 1205 ->
// 280; transposed 60x17x41x50 -> 48, 3x3 s2: 112 -> 57, 217x80x32x32 -> 96, 2x2 s2: 246 -> 201.
// Stores of 4 bytes were 14 - 25 % of the time: four pixels of a channel go together where a plane is whole fours (their
// pieces then have pixels in rows, channels in columns), two of neighbouring column phases where the stride is 2.
#include <cmath>
#include <type_traits>

#include "conv_f32.h"
#include "gemm_tile.h"

using namespace sofie;

namespace {

constexpr unsigned OUTSIDE = 0x40000000u;      // no descriptor of this file reaches it
constexpr unsigned NO_TAP = 0x80000000u;       // every lane's mask has this bit: an entry of the table that asks for nothing
constexpr int MAX_PHASES = 4;

struct AnyPhase {
   int P, PHW;                // pixels over all images, per image
   int KH, KW, sx, ph, pw;    // sx: floats the descriptor of x starts in front of the tensor
   int steps, last_steps;     // 4-k steps per block of CB channels, in the last block
   int table_steps;           // steps in front of the last block's in the table (0: there is one block)
   int groups16;              // 16-k groups over all of K (an even number: zeros behind K)
   int full_groups;           // groups whose steps all lie in full blocks
   int wofs;                  // first float of the phase's fragments
   int oy0, oys, ox0, oxs, OW;
   int th0, ths, tw0, tws;
   FastDiv dPHW, dOW, dKHW, dKW;
};

struct AnyArgs {
   const float *x, *w, *bias;
   float *y;
   unsigned xbytes, ybytes, wbytes;      // of this launch's images, of the fragments
   int H, W, icg, ocg, groups, sh, sw, dh, dw, relu;
   int CB, nblocks;
   int octiles;               // of 16 channels per group
   int oblocks;               // of TI tiles per group
   int chw4, hw4;             // bytes of an image, of a channel plane of x
   int ocplane4, plane4;      // bytes of an image, of a channel plane of y
   int OW0;
   int ks;                    // wavefronts that share the k of a tile
   FastDiv dOB;
   AnyPhase phase[MAX_PHASES];
};

struct TapEntry {
   unsigned off, tap;
};

// How a lane finds its values of x (above): no tap of the launch lies outside an image; a table of taps and a test per
// value; a table of the finished offsets.
enum { INSIDE, TESTED, LOOKED_UP };

typedef unsigned uint2_t __attribute__((ext_vector_type(2)));

// What a lane stores of a 16 x 16 piece: one pixel of four channels; four consecutive pixels of a channel with one
// instruction (they are in one plane); two neighbouring pixels of four channels, which come from the two column phases of
// a transposed convolution of stride 2: a wavefront sums one after the other.
enum { PIXELS, QUADS, PAIRS };

template <int TI, int TJ, int MODE, int STORE>
__global__ void __launch_bounds__(512, TI * TJ >= 10 || (TI * TJ == 8 && STORE == PAIRS) ? 3 : 4) k_conv_f32_any(AnyArgs g)
{
   ask_for_arguments<sizeof(g)>();
   extern __shared__ __align__(16) unsigned char smem_raw[];
   constexpr int NH = STORE == PAIRS ? 2 : 1;
   constexpr bool PAD = MODE == TESTED, LOOK = MODE == LOOKED_UP;
   TapEntry *const table = reinterpret_cast<TapEntry *>(smem_raw);
   auto phase_of = [&](int h) {
      AnyPhase q = g.phase[0];
#pragma unroll
      for (int i = 1; i < MAX_PHASES; ++i)
         if ((int)blockIdx.y * NH + h == i) q = g.phase[i];
      return q;
   };
   const AnyPhase q0 = phase_of(0);
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int r16 = lane & 15, kg = lane >> 4;
   const int waves = (int)blockDim.x >> 6;
   // workgroup id -> (pixels, channels): an XCD (an L2) works on consecutive ids, the channel blocks of a pixel block are
   // next to each other
   int pid = blockIdx.x;
   {
      const int tiles = gridDim.x, xcd = pid & 7, base = tiles >> 3, rem = tiles & 7;
      pid = (pid >> 3) + xcd * base + (xcd < rem ? xcd : rem);
   }
   const int pb = fdiv(pid, g.dOB), ob = pid - pb * g.oblocks * g.groups;
   const int grp = ob / g.oblocks, tile0 = (ob - grp * g.oblocks) * TI;
   const int strips = waves / g.ks, slice = wave % g.ks;
   const int px0 = (pb * strips + wave / g.ks) * 16 * TJ;
   if (pb * strips * 16 * TJ >= q0.P) return;      // the grid is as wide as the phase with most pixels

   v4f acc[NH][TI][TJ];
   // sums of one phase
   auto sum = [&](const AnyPhase &q, v4f (&acc)[TI][TJ]) {
   if constexpr (!LOOK) {
      // the table: entry e of a block is k = e; the last block's entries behind them; a step that asks for nothing
      const int KHW = q.KH * q.KW, main_len = 4 * q.table_steps, last_len = 4 * q.last_steps + 4;
      const int main_k = g.CB * KHW, last_k = (g.icg - (g.nblocks - 1) * g.CB) * KHW;
      for (int e = tid; e < main_len + last_len; e += (int)blockDim.x) {
         const int k = e < main_len ? e : e - main_len, ic = fdiv(k, q.dKHW), t = k - ic * KHW, a = fdiv(t, q.dKW), b = t - a * q.KW;
         const bool there = k < (e < main_len ? main_k : last_k);
         table[e] = there ? TapEntry{(unsigned)(ic * g.hw4 + (a * g.dh * g.W + b * g.dw) * 4), (1u << a) | (1u << (q.KH + b))}
                          : TapEntry{OUTSIDE, NO_TAP};
      }
   }
   // pixels of this lane: offset of the window's first cell, bits of the kernel rows and columns outside the image
   unsigned xofs[TJ], outside[PAD ? TJ : 1];
#pragma unroll
   for (int j = 0; j < TJ; ++j) {
      const int p = px0 + j * 16 + r16;
      const bool there = p < q.P;
      const int n = fdiv(there ? p : 0, q.dPHW), r = (there ? p : 0) - n * q.PHW, oy = fdiv(r, q.dOW), ox = r - oy * q.OW;
      xofs[j] = there ? (unsigned)(n * g.chw4 + (oy * g.sh * g.W + ox * g.sw) * 4) : OUTSIDE;
      if constexpr (PAD) {
         unsigned m = NO_TAP;
         for (int a = 0; a < q.KH; ++a) m |= (unsigned)(oy * g.sh - q.ph + a * g.dh) < (unsigned)g.H ? 0u : 1u << a;
         for (int b = 0; b < q.KW; ++b) m |= (unsigned)(ox * g.sw - q.pw + b * g.dw) < (unsigned)g.W ? 0u : 1u << (q.KH + b);
         outside[j] = there ? m : ~0u;
      }
      if constexpr (LOOK) {
         // [strip][tap][lane][j]; the wavefronts of a strip share the taps; behind the last tap one that asks for nothing
         unsigned *const mine = reinterpret_cast<unsigned *>(smem_raw) + ((wave / g.ks) * (q.KH * q.KW + 1) * 64 + lane) * TJ + j;
         const int iy = oy * g.sh - q.ph, ix = ox * g.sw - q.pw;
         for (int t = slice; t <= q.KH * q.KW; t += g.ks) {
            const int a = fdiv(t, q.dKW), b = t - a * q.KW;
            const bool in = there && a < q.KH && (unsigned)(iy + a * g.dh) < (unsigned)g.H && (unsigned)(ix + b * g.dw) < (unsigned)g.W;
            mine[t * 64 * TJ] = in ? xofs[j] + (unsigned)((a * g.dh * g.W + b * g.dw) * 4 + kg * g.hw4) : OUTSIDE;
         }
      }
   }
   __syncthreads();

   const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.x) - q.sx, 0, (int)(g.xbytes + 4 * q.sx), 0x00020000);
   const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.w) + q.wofs, 0, (int)(g.wbytes - 4 * q.wofs), 0x00020000);
   unsigned wofs[TI];         // uniform: fragments of this wavefront's tiles (those behind the last tile: the last one's)
#pragma unroll
   for (int i = 0; i < TI; ++i) {
      const int t = tile0 + i < g.octiles ? tile0 + i : g.octiles - 1;
      wofs[i] = (unsigned)__builtin_amdgcn_readfirstlane((grp * g.octiles + t) * q.groups16 * 1024);
   }
   const int per = ((q.groups16 + g.ks - 1) / g.ks + 1) & ~1;
   const int g0 = __builtin_amdgcn_readfirstlane(q.groups16 < slice * per ? q.groups16 : slice * per), g1 = __builtin_amdgcn_readfirstlane(q.groups16 < g0 + per ? q.groups16 : g0 + per);

   // where the loads are: block of channels, step of its table, first entry, uniform offset
   const unsigned *const offsets = reinterpret_cast<const unsigned *>(smem_raw) + ((wave / g.ks) * (q.KH * q.KW + 1) * 64 + lane) * TJ;
   const unsigned block4 = (unsigned)g.CB * (unsigned)g.hw4;
   int block, step, len, first;
   unsigned soff;
   auto go_to = [&](int group) {
      block = (4 * group) / q.steps;
      if (block > g.nblocks - 1) block = g.nblocks - 1;
      step = 4 * group - block * q.steps;
      len = block == g.nblocks - 1 ? q.last_steps : q.steps;
      if (step > len) step = len;
      first = block == g.nblocks - 1 ? 4 * q.table_steps : 0;
      soff = (unsigned)(grp * g.icg + block * g.CB) * (unsigned)g.hw4;
   };
   go_to(g0);

#pragma unroll
   for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

   struct Group {
      v4f w[TI];
      float x[4][TJ];
   };
   // FULL: every step of the group is one of a full block, so that the next step is a few scalar instructions without
   // branches; else it may be the last block's or lie behind the last step (the entry that asks for nothing)
   auto load = [&](Group &f, int gi, auto full) {
      constexpr bool FULL = decltype(full)::value;
#pragma unroll
      for (int i = 0; i < TI; ++i)
         f.w[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(wrs, lane * 16, (int)(wofs[i] + (unsigned)gi * 1024u), 0));
      unsigned v[4][TJ], so[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
         if constexpr (LOOK) {
            __builtin_memcpy(v[e], __builtin_assume_aligned(offsets + step * 64 * TJ, 4 * TJ), 4 * TJ);
         } else {
            const TapEntry t = table[(FULL ? 0 : first) + 4 * step + kg];
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
               v[e][j] = xofs[j] + t.off;
               if constexpr (PAD) v[e][j] = (outside[j] & t.tap) ? OUTSIDE : v[e][j];
            }
         }
         so[e] = soff;
         if constexpr (FULL) {
            const int inside = (step + 1 - q.steps) >> 31;      // -1, or 0 at the end of the block
            step = (step + 1) & inside;
            soff += block4 & ~(unsigned)inside;
         } else {
            const bool next = step + 1 == len && block + 1 < g.nblocks;
            step = next ? 0 : step < len ? step + 1 : len;
            block = next ? block + 1 : block;
            soff = next ? soff + block4 : soff;
            const bool last = block + 1 == g.nblocks;
            len = last ? q.last_steps : q.steps;
            first = last ? 4 * q.table_steps : 0;
         }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
         for (int j = 0; j < TJ; ++j)
            f.x[e][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)v[e][j], (int)so[e], 0));
   };
   auto multiply = [&](const Group &f) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
         for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
               acc[i][j] = STORE == QUADS ? __builtin_amdgcn_mfma_f32_16x16x4f32(f.x[e][j], f.w[i][e], acc[i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[i][e], f.x[e][j], acc[i][j], 0, 0, 0);
   };
   // (loads behind the slice are made and not used)
   Group fa, fb;
   load(fa, g0, std::false_type{});
   int gi = g0;
   for (; gi < g1 && gi + 2 < q.full_groups; gi += 2) {
      load(fb, gi + 1, std::true_type{});
      multiply(fa);
      __builtin_amdgcn_sched_barrier(0);
      load(fa, gi + 2, std::true_type{});
      multiply(fb);
      __builtin_amdgcn_sched_barrier(0);
   }
   go_to(gi + 1);
   for (; gi < g1; gi += 2) {
      load(fb, gi + 1, std::false_type{});
      multiply(fa);
      __builtin_amdgcn_sched_barrier(0);
      load(fa, gi + 2, std::false_type{});
      multiply(fb);
      __builtin_amdgcn_sched_barrier(0);
   }
   };
   sum(q0, acc[0]);
   if constexpr (NH == 2) {
      __syncthreads();      // the first phase's table is done with
      sum(phase_of(1), acc[NH - 1]);
   }

   const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(g.y, 0, (int)g.ybytes, 0x00020000);
   const rsrc_t yrs4 = make_rsrc(g.y, g.ybytes);
   auto finish = [&](float v, float b) {
      if (g.bias) v = __fadd_rn(v, b);
      return g.relu ? (v > 0.0f ? v : 0.0f) : v;
   };
   // one 16 x 16 piece (a uniform offset stays inside the descriptor's range)
   auto store = [&](v4f v, v4f v2, int i, int j) {
      const int oc = (tile0 + i) * 16;
      if (oc >= g.ocg) return;
      if constexpr (STORE == QUADS) {
         // pixels 4 * kg + e of channel r16
         const int p = px0 + j * 16 + 4 * kg, n = fdiv(p, q0.dPHW);
         const bool there = p < q0.P && oc + r16 < g.ocg;
         const float b = g.bias && there ? g.bias[grp * g.ocg + oc + r16] : 0.0f;
#pragma unroll
         for (int e = 0; e < 4; ++e) v[e] = finish(v[e], b);
         store16_buf(yrs4, v, there ? (unsigned)(n * g.ocplane4 + (p - n * q0.PHW) * 4 + r16 * g.plane4) : OUTSIDE,
                     (unsigned)(grp * g.ocg + oc) * (unsigned)g.plane4);
      } else {
         // channels 4 * kg + e of pixel r16
         const int p = px0 + j * 16 + r16, n = fdiv(p, q0.dPHW), r = p - n * q0.PHW, oy = fdiv(r, q0.dOW), ox = r - oy * q0.OW;
         const int column = q0.ox0 + ox * q0.oxs;
         const unsigned at = (unsigned)(n * g.ocplane4 + ((q0.oy0 + oy * q0.oys) * g.OW0 + column) * 4 + kg * 4 * g.plane4);
#pragma unroll
         for (int e = 0; e < 4; ++e) {
            if (oc + e >= g.ocg) continue;
            const bool there = p < q0.P && oc + 4 * kg + e < g.ocg;
            const float b = g.bias && there ? g.bias[grp * g.ocg + oc + 4 * kg + e] : 0.0f;
            const unsigned first = __builtin_bit_cast(unsigned, finish(v[e], b));
            const int soff = (int)((unsigned)(grp * g.ocg + oc + e) * (unsigned)g.plane4);
            if constexpr (STORE == PAIRS) {
               const uint2_t both = {first, __builtin_bit_cast(unsigned, finish(v2[e], b))};
               const bool two = there && column + 1 < g.OW0;
               __builtin_amdgcn_raw_buffer_store_b64(both, yrs, (int)(two ? at : OUTSIDE), soff, 0);
               if ((g.OW0 & 1) && there && !two) __builtin_amdgcn_raw_buffer_store_b32(first, yrs, (int)at, soff, 0);
            } else
               __builtin_amdgcn_raw_buffer_store_b32(first, yrs, (int)(there ? at : OUTSIDE), soff, 0);
         }
      }
   };
   if (g.ks == 1) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
         for (int j = 0; j < TJ; ++j) store(acc[0][i][j], acc[NH - 1][i][j], i, j);
      return;
   }
   if constexpr (NH * TI * TJ <= 8) {
      // sums of the wavefronts that share a tile, in the order of their k; 16 x 16 pieces dealt to them
      __syncthreads();      // the table is done with
      v4f *const red = reinterpret_cast<v4f *>(smem_raw);
      constexpr int PIECES = NH * TI * TJ;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
         for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) red[(wave * PIECES + (h * TI + i) * TJ + j) * 64 + lane] = acc[h][i][j];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
         for (int j = 0; j < TJ; ++j) {
            if ((i * TJ + j) % g.ks != slice) continue;
            v4f v[NH];
#pragma unroll
            for (int h = 0; h < NH; ++h) {
               v[h] = red[((wave - slice) * PIECES + (h * TI + i) * TJ + j) * 64 + lane];
               for (int s = 1; s < g.ks; ++s) {
                  const v4f u = red[((wave - slice + s) * PIECES + (h * TI + i) * TJ + j) * 64 + lane];
#pragma unroll
                  for (int e = 0; e < 4; ++e) v[h][e] = __fadd_rn(v[h][e], u[e]);
               }
            }
            store(v[0], v[NH - 1], i, j);
         }
   }
}

struct WeightArgs {
   const float *w;
   float *dst;
   int icg, ocg, octiles, CB, nblocks, quad, KH0, KW0, transposed, total4;      // quad: LOOKED_UP's order of k; total4: 16-byte pieces of all phases
   AnyPhase phase[MAX_PHASES];
};

// The fragments: 16 bytes per thread (lane's operands of four steps); zeros behind the last channel and the last k.
__global__ void __launch_bounds__(256) k_conv_f32_any_weights(WeightArgs g)
{
   const int idx = blockIdx.x * 256 + threadIdx.x;
   if (idx >= g.total4) return;
   AnyPhase q = g.phase[0];
#pragma unroll
   for (int i = 1; i < MAX_PHASES; ++i)
      if (g.phase[i].wofs > 0 && 4 * idx >= g.phase[i].wofs) q = g.phase[i];
   int r = idx - q.wofs / 4;
   const int lane = r & 63;
   r >>= 6;
   const int group = r % q.groups16;
   r /= q.groups16;
   const int tile = r % g.octiles, grp = r / g.octiles, oc = tile * 16 + (lane & 15);
   const int KHW = q.KH * q.KW;
   v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
   for (int e = 0; e < 4; ++e) {
      const int t = group * 4 + e;
      int b = t / q.steps;
      if (b > g.nblocks - 1) b = g.nblocks - 1;
      const int k = 4 * (t - b * q.steps) + (lane >> 4);
      const int icl = !g.quad ? fdiv(k, q.dKHW) : k < 4 * KHW ? lane >> 4 : g.icg, tap = !g.quad ? k - icl * KHW : k >> 2, ic = b * g.CB + icl;
      if (oc >= g.ocg || ic >= g.icg || (b < g.nblocks - 1 && icl >= g.CB)) continue;
      const int ta = fdiv(tap, q.dKW), a = q.th0 + ta * q.ths, c = q.tw0 + (tap - ta * q.KW) * q.tws;
      const size_t at = g.transposed ? ((size_t)(grp * g.icg + ic) * g.ocg + oc) : ((size_t)(grp * g.ocg + oc) * g.icg + ic);
      v[e] = g.w[(at * g.KH0 + a) * g.KW0 + c];
   }
   *reinterpret_cast<v4f *>(g.dst + (size_t)idx * 4) = v;
}

struct Form {
   int ti, tj, ks, store;
   double time;
};

// Time of a form in cycles. A wavefront needs for a group of 16 k what its matrix instructions (128 cycles a tile and group)
// or its requests (ten cycles of the compute unit each, less while SIMDs are idle) take, whichever is longer; the start
// and the loads' latency are shared by the wavefronts a SIMD holds; a store costs by its kind; the last round of wavefronts is
// not full. The constants are a fit to 200 convolutions over the ranges of perf/cases.py, timed in every form: the form this
// picks is 4 % behind the best of all forms in the mean, 29 % at most.
double estimate(const AnyArgs &g, int nphases, int cus, int mode, const Form &f)
{
   const double simds = 4.0 * cus, tiles = f.ti * f.tj, blocks = (double)g.groups * cdiv(g.octiles, f.ti);
   const int together = f.store == PAIRS ? 2 : 1;
   double waves = 0.0;
   for (int i = 0; i < nphases; i += together) waves += blocks * cdiv(g.phase[i].P, 16 * f.tj) * f.ks;
   const double per_simd = waves / simds;
   const double resident = tiles >= 10 || (f.store == PAIRS && tiles >= 8) ? 3 : tiles >= 8 ? 5 : tiles >= 4 ? 7 : 8;
   const double held = per_simd < 1 ? 1 : per_simd > resident ? resident : per_simd;
   const double busy = per_simd < 0.25 ? 0.25 : per_simd > 1 ? 1 : per_simd;
   const double mma = 128.0 * tiles + (mode == LOOKED_UP ? 45.0 : 161.0 * f.tj) + 4.0, requests = (188.0 * f.tj + 18.0 * f.ti) * busy;
   const double m2 = mma * mma, r2 = requests * requests, l2 = 148.0 * 148.0 / (held * held);
   const double group = std::sqrt(std::sqrt(m2 * m2 + r2 * r2 + l2 * l2));      // a smooth maximum
   double total = 0.0, longest = 0.0;
   for (int i = 0; i < nphases; i += together) {
      double wave = (f.ks > 1 ? 59.0 * tiles * together + 25.0 : 0.0) + tiles * (f.store == PAIRS ? 1610.0 : f.store == QUADS ? 645.0 : 1050.0) / f.ks;
      for (int h = 0; h < together; ++h) wave += ((cdiv(g.phase[i + h].groups16, f.ks) + 1) & ~1) * group + 5490.0 / held;
      total += wave * blocks * cdiv(g.phase[i].P, 16 * f.tj) * f.ks;
      if (wave > longest) longest = wave;
   }
   if (per_simd <= 1) return longest + 7550.0;
   return total / simds * (1.0 + 0.19 * (std::ceil(per_simd) - per_simd) / per_simd) + 7550.0;
}

template <int TI, int TJ, int STORE>
void (*form(int mode))(AnyArgs)
{
   if constexpr (STORE == PAIRS && TI * TJ > 8) {
      return nullptr;      // twice the accumulators
   } else {
      constexpr auto kern_i = k_conv_f32_any<TI, TJ, INSIDE, STORE>, kern_t = k_conv_f32_any<TI, TJ, TESTED, STORE>,
                     kern_l = k_conv_f32_any<TI, TJ, LOOKED_UP, STORE>;
      SOFIE_LARGE_LDS(kern_i);
      SOFIE_LARGE_LDS(kern_t);
      SOFIE_LARGE_LDS(kern_l);
      return mode == INSIDE ? kern_i : mode == TESTED ? kern_t : kern_l;
   }
}

template <int TI, int TJ>
int launch(sofie_hip_ctx *ctx, const AnyArgs &g, int nphases, int mode, int store, int ks, int tiles, size_t table_bytes)
{
   const auto kern = store == PAIRS ? form<TI, TJ, PAIRS>(mode) : store == QUADS ? form<TI, TJ, QUADS>(mode) : form<TI, TJ, PIXELS>(mode);
   if (store == PAIRS) nphases /= 2;
   const int waves = ks > 4 ? 8 : 4;
   if (mode == LOOKED_UP) table_bytes *= (size_t)(waves / ks) * TJ;      // given for a strip of 16 pixels
   const size_t sums = ks > 1 ? (size_t)waves * TI * TJ * (store == PAIRS ? 2048 : 1024) : 0;
   hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)nphases), dim3((unsigned)waves * 64),
                      table_bytes > sums ? table_bytes : sums, ctx->stream, g);
   return check_launch(ctx, "k_conv_f32_any");
}

}  // namespace

int sofie::conv_f32_any(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done, ConvWays ways)
{
   *done = false;
   const size_t image = (size_t)p.C * p.H * p.W * 4, out_image = (size_t)p.OC * p.OH0 * p.OW0 * 4;
   // descriptors and OUTSIDE: 1 GiB of images per launch, 16 MB less for what lies in front of the tensor
   const size_t room = ((size_t)1 << 30) - ((size_t)16 << 20);
   if (image > room || out_image > room || p.nphases < 1 || p.nphases > MAX_PHASES) return SOFIE_HIP_OK;
   // what may be stored together: pixels that are next to each other in whole fours of an image, or the column phases of
   // stride 2 (the second may have a column less)
   const ConvPhase &f0 = p.phase[0];
   const bool quads = p.nphases == 1 && f0.oys == 1 && f0.oxs == 1 && f0.oy0 == 0 && f0.ox0 == 0 && f0.OW == p.OW0 && f0.OH == p.OH0 &&
                      p.OH0 * p.OW0 % 4 == 0;
   bool pairs = f0.oxs == 2 && p.nphases % 2 == 0;
   for (int i = 0; pairs && i < p.nphases; i += 2) {
      const ConvPhase &a = p.phase[i], &b = p.phase[i + 1];
      pairs = a.ox0 == 0 && b.ox0 == 1 && a.oy0 == b.oy0 && a.OH == b.OH && b.OW <= a.OW;
   }
   AnyArgs g{};
   g.icg = p.C / p.groups;
   g.ocg = p.OC / p.groups;
   g.octiles = cdiv(g.ocg, 16);
   bool pad = false;
   int max_taps = 0;
   bool bits = true;      // a bit per kernel row and column and one for NO_TAP
   for (int i = 0; i < p.nphases; ++i) {
      const ConvPhase &f = p.phase[i];
      if (f.KH < 1 || f.KW < 1 || f.OH < 1 || f.OW < 1) return SOFIE_HIP_OK;
      if ((long)f.KH * f.KW > (1 << 16)) return SOFIE_HIP_OK;
      if (f.KH * f.KW > max_taps) max_taps = f.KH * f.KW;
      bits = bits && f.KH + f.KW <= 31;
      const long front = (long)f.ph * p.W + f.pw;
      if (front > (1 << 21) || (front < 0 && -front >= (long)p.H * p.W)) return SOFIE_HIP_OK;
      // (a pair sums as many columns of the second phase as of the first)
      const int columns = pairs ? p.phase[i & ~1].OW : f.OW;
      pad = pad || f.ph > 0 || f.pw > 0 || (long)(f.OH - 1) * p.sh - f.ph + (long)(f.KH - 1) * p.dh >= p.H ||
            (long)(columns - 1) * p.sw - f.pw + (long)(f.KW - 1) * p.dw >= p.W;
      // a window that starts behind the tensor's first cell and one whose offsets leave 32 bits stay with the general kernel
      if (((long)(f.KH - 1) * p.dh * p.W + (long)(f.KW - 1) * p.dw) * 4 > (long)room / 2) return SOFIE_HIP_OK;
      if ((((long)(f.OH - 1) * p.sh + 1) * p.W + (long)(columns - 1) * p.sw) * 4 > (long)room) return SOFIE_HIP_OK;
   }
   // Finished offsets where four channels go with each tap and the table (taps x 256 bytes per 16 pixels) is short: no vector
   // arithmetic per value (256x64x56x56 -> 128, 3x3: 900 us against 972 with the test; 256x64x10x10 -> 128: 45 against 49).
   // Else all channels in one table where that is short (no step is cut off at a block's end), or four at a time (whole
   // steps for any kernel).
   // (Very long kernels have no bit per row and column: finished offsets as long as they fit the LDS.)
   const bool quad = g.icg % 4 == 0 && max_taps <= (bits || !pad ? 12 : 96);
   if (!quad && pad && !bits) return SOFIE_HIP_OK;
   g.CB = !quad && (long)g.icg * max_taps <= 640 ? g.icg : 4;
   g.nblocks = cdiv(g.icg, g.CB);
   size_t wfloats = 0, table_bytes = 0;
   for (int i = 0; i < p.nphases; ++i) {
      const ConvPhase &f = p.phase[i];
      AnyPhase &q = g.phase[i];
      const int KHW = f.KH * f.KW;
      q.KH = f.KH; q.KW = f.KW; q.ph = f.ph; q.pw = f.pw;
      q.sx = f.ph * p.W + f.pw;
      q.steps = g.nblocks > 1 || quad ? KHW : cdiv(g.icg * KHW, 4);
      q.last_steps = cdiv((g.icg - (g.nblocks - 1) * g.CB) * KHW, 4);
      q.table_steps = g.nblocks > 1 ? q.steps : 0;
      const long steps = (long)(g.nblocks - 1) * q.steps + q.last_steps;
      if (steps > (1 << 24)) return SOFIE_HIP_OK;
      q.groups16 = (cdiv((int)steps, 4) + 1) & ~1;      // the loop takes two at a time
      q.full_groups = (int)(g.nblocks > 1 && g.icg % g.CB ? (long)(g.nblocks - 1) * q.steps : steps) / 4;
      q.wofs = (int)wfloats;
      const size_t floats = (size_t)p.groups * g.octiles * q.groups16 * 256;
      wfloats += floats;
      if (wfloats * 4 > room / 2) return SOFIE_HIP_OK;
      q.oy0 = f.oy0; q.oys = f.oys; q.ox0 = f.ox0; q.oxs = f.oxs;
      q.th0 = f.th0; q.ths = f.ths; q.tw0 = f.tw0; q.tws = f.tws;
      q.dKHW = make_fastdiv((unsigned)KHW);
      q.dKW = make_fastdiv((unsigned)f.KW);
      if ((long)q.table_steps + q.last_steps > 4096) return SOFIE_HIP_OK;
      const size_t table = quad ? (size_t)(KHW + 1) * 256 : (size_t)(q.table_steps + q.last_steps + 1) * 4 * sizeof(TapEntry);
      if (table > table_bytes) table_bytes = table;
   }
   // three groups behind the last fragment may be asked for, to no use
   const size_t wbytes = wfloats * 4 + 4096;
   g.wbytes = (unsigned)wbytes;
   // images per launch
   size_t per = room / (image > out_image ? image : out_image);
   for (int i = 0; i < p.nphases; ++i)
      if (per * p.phase[i & ~1].OW * p.phase[i].OH > ((size_t)1 << 30)) per = ((size_t)1 << 30) / ((size_t)p.phase[i & ~1].OW * p.phase[i].OH);
   if (per > (size_t)p.N) per = (size_t)p.N;
   if (per < 1) return SOFIE_HIP_OK;

   const int mode = quad ? LOOKED_UP : pad ? TESTED : INSIDE;
   g.groups = p.groups;
   const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
   // the form for a launch on n images, and the pixels of g for it
   auto choose = [&](size_t n) {
      // the pixels a form works on: those of each phase, or in a pair as many columns in both
      auto set_pixels = [&](int store) {
         for (int i = 0; i < p.nphases; ++i) {
            AnyPhase &q = g.phase[i];
            q.OW = p.phase[store == PAIRS ? i & ~1 : i].OW;
            q.PHW = p.phase[i].OH * q.OW;
            q.P = (int)n * q.PHW;
            q.dPHW = make_fastdiv((unsigned)q.PHW);
            q.dOW = make_fastdiv((unsigned)q.OW);
         }
      };
      // Pairs where a phase is a short sum and its output is large: the time is the stores' then (66x33x37x37 -> 64, 2x2: 56 us in
      // pairs, 67 pixel by pixel); else the phases side by side (64x128x28x28 -> 64, 4x4: 122 against 132; small layers:
      // half the wavefronts).
      int store = quads ? QUADS : PIXELS;
      if (pairs) {
         long k = 0, pixels = 0;
         for (int i = 0; i < p.nphases; ++i) {
            k += (long)g.icg * g.phase[i].KH * g.phase[i].KW;
            pixels += (long)p.phase[i].OH * p.phase[i].OW;
         }
         if (k <= 112 * p.nphases && (double)n * p.OC * pixels >= 8e6) store = PAIRS;
      }
      set_pixels(store);
      static const int forms[][2] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {3, 2}, {4, 2}, {5, 2}, {6, 2}};
      Form best{0, 0, 0, store, 0.0};
      for (const auto &f : forms)
         for (int ks = 1; ks <= 8; ks *= 2) {
            const int tiles = f[0] * f[1];
            if ((f[0] > g.octiles && f[0] > 1) || (ks > 1 && ks > g.phase[0].groups16)) continue;      // tiles or wavefronts of nothing
            // the sums of wavefronts that share a tile go through the LDS; a pair has twice the accumulators; 4-byte stores of
            // many tiles in a row hold up everybody (64x128x28x28 -> 64: 132 us with four tiles of channels, 124 with two)
            if (ks > 1 && (tiles * ks > 32 || tiles * (store == PAIRS ? 2 : 1) > 8)) continue;
            if (store == PAIRS ? tiles > 8 : p.nphases > 1 && f[0] > 3) continue;
            if (quad && table_bytes * ((ks > 4 ? 8 : 4) / ks) * f[1] > (size_t)kMaxDynamicLds) continue;
            Form form{f[0], f[1], ks, store, 0.0};
            form.time = estimate(g, p.nphases, cus, mode, form);
            if (best.ti == 0 || form.time < best.time) best = form;
         }
      return best;
   };
   Form best = choose(per);
   if (best.ti == 0) return SOFIE_HIP_OK;
   const double here_us = best.time / 2400.0 * ((double)p.N / (double)per) + (ctx->constant_weights ? 0.0 : 3.1);
   // Shorter sums are shorter on the vector unit.
   if (ways != SPLIT_ONLY)
      if (int rc = conv_f32_short(ctx, p, 0.9 * (here_us < other_us ? here_us : other_us), done); rc || *done) return rc;
   // Longer sums on many tiles are shorter on the bf16 matrix instructions. The estimates are off by some 10 %; of 42 random 3x3 layers of 18 to
   // 26 channels that it takes none is longer than on the kernel it takes the place of.
   if (ways != SPLIT_DECLINED)
      if (int rc = conv_f32_split(ctx, p, 0.9 * here_us < 0.95 * other_us ? 0.9 * here_us : 0.95 * other_us, done); rc || *done) return rc;
   if (ways == SPLIT_ONLY) return SOFIE_HIP_OK;
   // against what the caller has instead (the estimate's unit is a cycle at 2400 MHz; weights that are not kept are laid out in
   // front of the launch, 3.1 us)
   if (other_us < 0.95 * here_us) return SOFIE_HIP_OK;

   int key[8 + 7 * MAX_PHASES] = {quad ? 4 : 3, p.groups, g.ocg, g.icg, p.KH0, p.KW0, p.transposed, p.nphases};
   for (int i = 0; i < p.nphases; ++i) {
      const AnyPhase &q = g.phase[i];
      const int v[7] = {q.KH, q.KW, q.th0, q.ths, q.tw0, q.tws, q.wofs};
      for (int e = 0; e < 7; ++e) key[8 + 7 * i + e] = v[e];
   }
   void *ws = nullptr;
   bool fresh = true;
   // (while a graph is recorded the scratch buffer may be too small: the general kernel needs none)
   if (packed_weights(ctx, p.w, layout_key(key, 8 + 7 * p.nphases), wbytes, &ws, &fresh)) return SOFIE_HIP_OK;
   if (fresh) {
      WeightArgs a{};
      a.w = p.w; a.dst = static_cast<float *>(ws);
      a.icg = g.icg; a.ocg = g.ocg; a.octiles = g.octiles; a.CB = g.CB; a.nblocks = g.nblocks; a.quad = quad;
      a.KH0 = p.KH0; a.KW0 = p.KW0; a.transposed = p.transposed; a.total4 = (int)(wfloats / 4);
      for (int i = 0; i < MAX_PHASES; ++i) a.phase[i] = g.phase[i];
      hipLaunchKernelGGL(k_conv_f32_any_weights, dim3((unsigned)cdiv(a.total4, 256)), dim3(256), 0, ctx->stream, a);
      if (int rc = check_launch(ctx, "k_conv_f32_any_weights")) return rc;
   }
   g.w = static_cast<const float *>(ws);
   g.bias = p.bias;
   g.H = p.H; g.W = p.W; g.sh = p.sh; g.sw = p.sw; g.dh = p.dh; g.dw = p.dw; g.relu = p.relu;
   g.chw4 = (int)image;
   g.hw4 = p.H * p.W * 4;
   g.ocplane4 = (int)out_image;
   g.plane4 = p.OH0 * p.OW0 * 4;
   g.OW0 = p.OW0;
   for (size_t n0 = 0; n0 < (size_t)p.N; n0 += per) {
      const size_t n = (size_t)p.N - n0 < per ? (size_t)p.N - n0 : per;
      g.x = p.x + n0 * (image / 4);
      g.y = p.y + n0 * (out_image / 4);
      g.xbytes = (unsigned)(n * image);
      g.ybytes = (unsigned)(n * out_image);
      if (n != per) best = choose(n);
      g.ks = best.ks;
      g.oblocks = cdiv(g.octiles, best.ti);
      g.dOB = make_fastdiv((unsigned)(g.oblocks * g.groups));
      const int waves = best.ks > 4 ? 8 : 4, strips = waves / best.ks;
      long tiles = 0;
      for (int i = 0; i < p.nphases; ++i) {
         const long t = (long)cdiv(g.phase[i].P, 16 * best.tj * strips) * g.oblocks * g.groups;
         if (t > tiles) tiles = t;
      }
      if (tiles > ((long)1 << 30)) return set_error(ctx, SOFIE_HIP_EINVAL, "%s: too many tiles", __func__);
      int rc = SOFIE_HIP_OK;
      switch (best.ti * 10 + best.tj) {
#define SOFIE_FORM(i, j) case i * 10 + j: rc = launch<i, j>(ctx, g, p.nphases, mode, best.store, best.ks, (int)tiles, table_bytes); break
         SOFIE_FORM(1, 1); SOFIE_FORM(2, 1); SOFIE_FORM(1, 2); SOFIE_FORM(2, 2); SOFIE_FORM(3, 2); SOFIE_FORM(4, 2); SOFIE_FORM(5, 2);
         SOFIE_FORM(6, 2);
#undef SOFIE_FORM
      }
      if (rc) return rc;
   }
   *done = true;
   return SOFIE_HIP_OK;
}
