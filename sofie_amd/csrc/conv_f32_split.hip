// fp32 NCHW convolutions of any channels, kernels, strides, dilations and groups, and the output phases of transposed ones, as an
// implicit GEMM on the bf16 matrix instructions with every operand as three bf16 numbers (split_bf16.h): k_conv_f32_split.
//
//   Y[oc, pixel] = sum_k W[oc, k] * X[k, pixel],  k = (8 channels, kernel row, kernel column, channel of the 8)
//
// A workgroup of four wavefronts (2 x 2) owns 32 TI channels x 32 TJ pixels, a wavefront TI x TJ tiles of 16 x 16.
//   * X: the input cells of the tile's pixels (halo included, zeros outside the image) lie in LDS as h, m, l of eight channels
//     each, 48 bytes a cell, CS channels (a slot) at a time: a cell is split once and read by all taps. 16 lanes with neighbouring
//     cells fall on different banks, at stride 2, too. Two slots: while one is multiplied the threads hold the loads of the slot
//     after the next in registers; behind a barrier they convert them and put them where the finished slot was. A step of 32 k is
//     four chunks of 8 channels of a tap, in one list over all slots, so that no step is cut off at a slot's end (9 taps of 16
//     channels are 4 1/2 steps); a step that reaches into the next slot has a barrier of its own.
//   * W: a copy laid out as fragments of split numbers [16 channels][step][h, m, l][lane], once per tensor under the
//     constant-weights promise, else in front of the launch. Straight into registers, a step ahead.
//   * Pixels run over all images in one row, or, where that costs little, tiles end with an image; wide images are cut into strips.
// Few channels and a large kernel (ROWS; the first layer of an image network): eight channels of a cell would be mostly zeros. There a cell
// is the eight values that a row of the kernel meets at an output column, of one channel; a chunk of K is a row of the kernel, zeros up
// to eight columns, K = (channel, kernel row, kernel column) in one slot. A value is split once per output column it
// is read at, still shared by the kernel's rows. Loaded as two 16-byte pieces from any dword; columns outside the image are zeroed behind
// the load. 16x3x224x224 -> 64, 7x7 s2 52.6 -> 33.2 us (k_conv_f32_any, 53 % of the fp32 instructions' rate); 53 of 90 random layers of
// one to five channels and kernels of 4 to 7 columns, 1.3 times shorter in the mean (55x5x38x38 -> 146, 7x7 s2 35.9 -> 16.9; 126x1x66x66 ->
// 54, 7x7 66.8 -> 43.4). Relative error against 64 bits 5e-8 to 9e-8 (1.1e-7 to 3.1e-7 before).
// Strips of an image take turns: neighbouring ones write halves of the same 128-byte lines, which one behind the other meet in an
// L2 (88x1x96x96 -> 150, 7x7 in strips of 16 columns 248 us strip by strip, 192 in turns).
// The four phases of a transposed layer of stride 2 x 2 (TOGETHER): a workgroup for each of them reads and splits the same cells and
// stores every other column. Here a workgroup has a wavefront for each phase on 16 TJ places of one patch; where rows are whole fours two phases
// exchange half of their columns in LDS and store 16 bytes each. What bounds it then are the weights, 12 KB a step and wavefront from
// the L2 where four wavefronts share them otherwise. Transposed 64x128x28x28 -> 64, 4x4 s2 89.5 -> 81; 140 random layers of stride 2 1.1 times
// shorter in the mean, 1.2 to 1.6 times where the route changed (3x3, 56x107x56x56 -> 16 97 -> 68.5; 2x2, 114x231x48x35 -> 16 136 -> 104).
// A layer of stride 2 reads four cells a pixel: slots of eight channels (choose_eights), whose odd number of chunks makes whole steps over four slots.
// 33x128x99x99 -> 128, 3x3 s2 244 us on k_conv_f32_any, 170 here; 48x80x144x11 -> 192, 7x7 s2 331, 167; 45 of 100 random layers of stride 2 1.1 to 2 times shorter,
// the others unchanged.
// All requests of a slot leave in one step: the fragments behind them wait for them (loads return in order), and one such wait
// per slot is cheaper than one per step. A bias read behind the loop made the compiler wait for each store in front of the next one
// (13000 cycles for 16 stores instead of 6800).
//
// Bound: the device's power under bf16 matrix instructions on large layers (256x64x56x56 -> 128: 1.65 GHz, the matrix pipe
// busy for 60 to 70 % of the cycles; without any loads in the loop 458 us), prologue, slots' waits and stores on
// smaller ones. Relative error against 64 bits a quarter of the fp32 instructions'. us against k_conv_f32_any and k_conv2d_f32_dma:
// 256x64x56x56 -> 128, 3x3 906 -> 568; 256x32x20x20 -> 64 47.4 -> 29.4; 256x64x10x10 -> 128 44.4 -> 27.2; 169x80x16x16 -> 128,
// 5x5 220 -> 102; 16x64x32x32 -> 65, 7x7 107 -> 49.5; transposed 64x128x28x28 -> 64, 4x4 s2 123 -> 81. Three workgroups per compute
// unit instead of two (fewer cells per thread and slot) were 12 % of the last.
#include "conv_f32.h"
#include "conv_f32_split_plan.h"
#include "gemm_tile.h"
#include "split_bf16.h"

using namespace sofie;

namespace {

constexpr unsigned OUTSIDE = 0x40000000u;      // no descriptor of this file reaches it
constexpr int MAX_PHASES = SplitPlan::MAX_PHASES, CELL = SplitPlan::CELL, THREADS = SplitPlan::THREADS;
static_assert(SplitPlan::MAX_LDS == kMaxDynamicLds, "LDS of a compute unit");

struct SplitPhase {
   int P, PHW, panels;        // pixels, of a panel; panels (strips of images)
   int ws, strips;            // columns of a strip, strips of an image
   int KH, KW, ph, pw;
   int HP, PW, cells;         // rows of a panel's input, cells of a row, of a tile's patch
   int full;                  // pixels of a panel that exist (PHW: up to whole tiles where tiles do not run on into the next panel)
   int chunks;                // of a slot: 8 channels of a tap each
   int steps;                 // of four chunks, all of K
   int wofs;                  // first 16-byte piece of the phase's fragments
   int OW;
   int oy0, oys, ox0, oxs;
   int th0, ths, tw0, tws;
   int tiles;                 // of a panel, where it is whole tiles and not the only one of its image: strips take turns; else 0
   FastDiv dTiles, dPHW, dWS, dHP, dPW, dStrips, dTaps, dKW, dCells;
   int ring;                  // chunks of two slots, or of four (an odd number of chunks): whole steps
   int down, right;           // TOGETHER: where its taps begin in the patch, whose pads are ph and pw
   int OH;
};

struct SplitArgs {
   const float *x, *w0, *bias;      // w0: the weights as they were given
   const v4i *w;
   float *y;
   unsigned xbytes, ybytes, wbytes;
   int H, W, icg, ocg, groups, KH0, KW0, transposed, sh, sw, dh, dw, relu;
   int CS, nslots;            // channels of a slot, slots
   int octiles, oblocks;
   int chw4, hw4, ocplane4, plane4, OW0;
   int table_bytes, slot_bytes;      // LDS: table of offsets, two slots
   int nphases;
   FastDiv dOB, dPhases;
   SplitPhase phase[MAX_PHASES];
   int table_ints;            // TOGETHER: from one phase's table to the next one's
};

enum { PIXELS, QUADS };
typedef float v2f __attribute__((ext_vector_type(2)));

// Where the caller's weight of a phase's tap (a, b) lies.
template <class Args>
__device__ __forceinline__ unsigned weight_at(const Args &g, const SplitPhase &q, int grp, int oc, int ic, int a, int b, bool rows)
{
   const int at = g.transposed ? (grp * g.icg + ic) * g.ocg + oc : (grp * g.ocg + oc) * g.icg + ic;
   return (unsigned)((at * g.KH0 + q.th0 + a * q.ths) * g.KW0 + (rows ? b : q.tw0 + b * q.tws));
}

// WO: wavefronts along the channels; TOGETHER: all have the same channels and pixels, of a phase each
template <int TI, int TJ, int WO, int STORE, bool PHASES, bool ROWS>
__global__ void __launch_bounds__(THREADS, SplitPlan::resident_of(TI, TJ, WO)) k_conv_f32_split(SplitArgs g)
{
   extern __shared__ __align__(16) unsigned char smem_raw[];
   constexpr bool TOGETHER = WO == SplitPlan::TOGETHER;
   if constexpr (PHASES || TOGETHER) ask_for_arguments<sizeof(g)>();
   constexpr int BP = 4 / WO * TJ * 16, ITEMS = SplitPlan::items_of(TI, TJ, WO, ROWS);
   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int r16 = lane & 15, kg = lane >> 4, wp = wave / WO, wo = TOGETHER ? 0 : wave % WO;
   // workgroup id -> (pixels, channels, phase): an XCD (an L2) works on consecutive ids; the phases of a tile, which read the same
   // input and write every other pixel of the same lines, are next to each other, and so are the channel blocks of a pixel block
   int pid = blockIdx.x, phase = 0;
   {
      const int tiles = gridDim.x, xcd = pid & 7, base = tiles >> 3, rem = tiles & 7;
      pid = (pid >> 3) + xcd * base + (xcd < rem ? xcd : rem);
   }
   if constexpr (TOGETHER) {
      phase = wave ^ (pid & 3);      // (phases of unequal length on every SIMD)
   } else if constexpr (PHASES) {
      const int all = pid;
      pid = fdiv(all, g.dPhases);
      phase = all - pid * g.nphases;
   }
   SplitPhase q = g.phase[0];
   if constexpr (PHASES || TOGETHER) {
#pragma unroll
      for (int i = 1; i < MAX_PHASES; ++i)
         if (phase == i) q = g.phase[i];
   }
   int pb = fdiv(pid, g.dOB);
   const int ob = pid - pb * g.oblocks * g.groups;
   if (q.tiles > 0) {         // (n, tile, strip) -> (n, strip, tile)
      const int n = fdiv(pb, q.dTiles), r = pb - n * q.strips * q.tiles, t = fdiv(r, q.dStrips);
      pb = (n * q.strips + r - t * q.strips) * q.tiles + t;
   }
   const int grp = ob / g.oblocks, tile0 = (ob - grp * g.oblocks) * TI * (TOGETHER ? 1 : WO) + wo * TI;
   const int p0 = pb * BP;
   if (p0 >= q.P) return;
   int origin;      // the tile's first row of the panels' inputs
   {
      const int panel = fdiv(p0, q.dPHW);
      origin = panel * q.HP + fdiv(p0 - panel * q.PHW, q.dWS) * g.sh;
   }
   unsigned char *const patch = smem_raw + g.table_bytes;
   unsigned voff[ITEMS];
   int column[ITEMS];         // ROWS: of the cell's first value
   const int items = q.cells * (g.CS >> 3);
#pragma unroll
   for (int s = 0; s < ITEMS; ++s) {
      const int item = s * THREADS + tid, c8 = fdiv(item, q.dCells), cell = item - c8 * q.cells, row = fdiv(cell, q.dPW), col = cell - row * q.PW;
      const int grow = origin + row, panel = fdiv(grow, q.dHP), n = fdiv(panel, q.dStrips);
      const int iy = grow - panel * q.HP - q.ph, ix = ((panel - n * q.strips) * q.ws + (ROWS ? col : 0)) * g.sw + (ROWS ? 0 : col) - q.pw;
      if constexpr (ROWS) {
         const bool row_there = item < items && panel < q.panels && (unsigned)iy < (unsigned)g.H;
         column[s] = row_there ? ix : -(1 << 28);
         voff[s] = row_there ? (unsigned)(n * g.chw4 + (iy * g.W + ix) * 4 + (grp * g.icg + c8) * g.hw4) : OUTSIDE;
         continue;
      }
      const bool in = item < items && panel < q.panels && (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W;
      voff[s] = in ? (unsigned)(n * g.chw4 + (iy * g.W + ix) * 4 + c8 * 8 * g.hw4) : OUTSIDE;
   }
   const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.x), 0, (int)g.xbytes, 0x00020000);
   const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4i *>(g.w) + q.wofs, 0, (int)(g.wbytes - 16u * (unsigned)q.wofs), 0x00020000);
   float xr[ITEMS][8];
   auto fetch = [&](float (&xr)[ITEMS][8], int s, int slot) {
      const int c0 = slot * g.CS, rem = g.icg - c0;
      const unsigned soff = (unsigned)(grp * g.icg + c0) * (unsigned)g.hw4;
      if (rem >= g.CS) {
#pragma unroll
         for (int e = 0; e < 8; ++e)
            xr[s][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)voff[s], (int)(soff + e * (unsigned)g.hw4), 0));
      } else {
         // channels behind the group's last one ask for nothing
         const int left = rem - fdiv(s * THREADS + tid, q.dCells) * 8;
#pragma unroll
         for (int e = 0; e < 8; ++e)
            xr[s][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)(e < left ? voff[s] : OUTSIDE), (int)(e < rem ? soff + e * (unsigned)g.hw4 : 0u), 0));
      }
   };
   // ROWS: eight values of a row at once, those that are not there (and where a cell begins in front of the tensor or ends behind
   // it, each by itself); put() leaves the columns of the image and of the kernel
   auto fetch_rows = [&](float (&xr)[ITEMS][8]) {
      bool edge = g.dw != 1;
#pragma unroll
      for (int s = 0; s < ITEMS; ++s) edge |= (int)voff[s] < 0 || (voff[s] != OUTSIDE && voff[s] + 32u > g.xbytes);
      if (__builtin_amdgcn_ballot_w64(edge) != 0) {
#pragma unroll
         for (int s = 0; s < ITEMS; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e)
               xr[s][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)((unsigned)(column[s] + e * g.dw) < (unsigned)g.W ? voff[s] + (unsigned)(e * g.dw * 4) : OUTSIDE), 0, 0));
         return;
      }
#pragma unroll
      for (int s = 0; s < ITEMS; ++s)
#pragma unroll
         for (int h = 0; h < 2; ++h) {
            const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)voff[s], 16 * h, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) xr[s][4 * h + e] = v[e];
         }
   };
   auto put = [&](const float (&xr)[ITEMS][8], int s, unsigned char *buf) {
      if (s * THREADS + tid >= items) return;
      v4i v[3];
      if constexpr (ROWS) {
         float there[8];
#pragma unroll
         for (int e = 0; e < 8; ++e) there[e] = e < q.KW && (unsigned)(column[s] + e * g.dw) < (unsigned)g.W ? xr[s][e] : 0.0f;
         split8(there, v);
      } else {
         split8(xr[s], v);
      }
      v4i *const d = reinterpret_cast<v4i *>(buf + (s * THREADS + tid) * CELL);
      d[0] = v[0];
      d[1] = v[1];
      d[2] = v[2];
   };
   unsigned wofs[TI];         // uniform: fragments of this wavefront's tiles (those behind the last tile: the last one's)
#pragma unroll
   for (int i = 0; i < TI; ++i) {
      const int t = tile0 + i < g.octiles ? tile0 + i : g.octiles - 1;
      wofs[i] = (unsigned)__builtin_amdgcn_readfirstlane((grp * g.octiles + t) * q.steps * 3072);
   }
   v8b w[TI][3];
   auto load_w = [&](int i, unsigned step) {
#pragma unroll
      for (int p = 0; p < 3; ++p)
         w[i][p] = __builtin_bit_cast(v8b, __builtin_amdgcn_raw_buffer_load_b128(wrs, lane * 16 + p * 1024, (int)(wofs[i] + step * 3072u), 0));
   };
   // everything that comes from memory is requested first; what the loop needs besides is worked out while it travels
   float second[ITEMS][8];
   if constexpr (ROWS) {
      fetch_rows(xr);
   } else {
#pragma unroll
      for (int s = 0; s < ITEMS; ++s)
         if (s * THREADS < items) fetch(xr, s, 0);
   }
   if (!ROWS && g.nslots > 1) {
#pragma unroll
      for (int s = 0; s < ITEMS; ++s)
         if (s * THREADS < items) fetch(second, s, 1);
   }
#pragma unroll
   for (int i = 0; i < TI; ++i) load_w(i, 0);
   constexpr int NB = STORE == QUADS ? 1 : 4;
   float bias[TI][NB];
#pragma unroll
   for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int e = 0; e < NB; ++e) {
         const int oc = (tile0 + i) * 16 + (STORE == QUADS ? r16 : 4 * kg + e);
         bias[i][e] = g.bias && oc < g.ocg ? g.bias[grp * g.ocg + oc] : 0.0f;
      }
   __builtin_amdgcn_sched_barrier(0);
   const int taps = q.KH * q.KW;
   int *const table = reinterpret_cast<int *>(smem_raw) + (TOGETHER ? phase * g.table_ints : 0);
   const int ring = ROWS ? 2 * q.chunks : q.ring, down = TOGETHER ? q.down : 0, right = TOGETHER ? q.right : 0;
   // offset of every chunk of two slots, or of four (chunks behind K, whose weights are zeros, read what lies in the slot: where there is one, its
   // first chunks)
   for (int e = TOGETHER ? lane : tid; e < ring; e += TOGETHER ? 64 : THREADS) {
      const int slot = (e >= q.chunks) + (ROWS ? 0 : (e >= 2 * q.chunks) + (e >= 3 * q.chunks)), second = slot & 1, k = e - slot * q.chunks, c8 = fdiv(k, q.dTaps), t = k - c8 * (ROWS ? q.KH : taps), a = ROWS ? t : fdiv(t, q.dKW), b = ROWS ? 0 : t - a * q.KW;
      table[e] = (c8 * q.cells + a * g.dh * q.PW + b * g.dw) * CELL + (g.nslots > 1 ? second * g.slot_bytes : 0);
   }
   int base[TJ];
#pragma unroll
   for (int j = 0; j < TJ; ++j) {
      const int p = p0 + (wp * TJ + j) * 16 + r16, panel = fdiv(p, q.dPHW), r = p - panel * q.PHW, oy = fdiv(r, q.dWS), c = r - oy * q.ws;
      base[j] = p < q.P && r < q.full ? ((panel * q.HP + oy * g.sh + down - origin) * q.PW + (ROWS ? c : c * g.sw) + right) * CELL : 0;
   }
   v4f acc[TI][TJ];
#pragma unroll
   for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
   for (int s = 0; s < ITEMS; ++s)
      if (s * THREADS < items) put(xr, s, patch);
   if (!ROWS && g.nslots > 1) {
#pragma unroll
      for (int s = 0; s < ITEMS; ++s)
         if (s * THREADS < items) put(second, s, patch + g.slot_bytes);
   }
   // (settled here: behind the loop the compiler would wait for the stores in front of each use)
#pragma unroll
   for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int e = 0; e < NB; ++e) asm volatile("" : "+v"(bias[i][e]));
   __syncthreads();
   int step = 0, place = 0;      // place: first chunk of the step in the table
   v8b x[TJ][3];
   auto read_x = [&](int j, int off) {
#pragma unroll
      for (int p = 0; p < 3; ++p) x[j][p] = *reinterpret_cast<const v8b *>(patch + base[j] + off + p * 16);
   };
   for (int slot = 0; slot < g.nslots; ++slot) {
      const bool last = ROWS || slot + 1 == g.nslots, more = !ROWS && slot + 2 < g.nslots;
      const int end_chunk = q.chunks * (slot + 1), end = last ? q.steps : (end_chunk + 3) >> 2;
      const bool across = !last && (end_chunk & 3) != 0;      // the last step takes chunks of the next slot, too
      const int begin = step;
      bool fresh = true;
      for (; step < end; ++step) {
         if (across && step + 1 == end) {
            __syncthreads();
            fresh = true;
         }
         if (fresh) {
            const int off = table[place + kg];
#pragma unroll
            for (int j = 0; j < TJ; ++j) read_x(j, off);
         }
         place = place + 4 == ring ? 0 : place + 4;
         const int ahead = across ? end - 2 : end - 1;
         fresh = step >= ahead;
         const int off = table[(fresh ? 0 : place) + kg];
         if (more && step == begin) {
#pragma unroll
            for (int s = 0; s < ITEMS; ++s)
               if (s * THREADS < items) fetch(xr, s, slot + 2);
         }
         // The six products of a tile one behind the other (17 cycles each; 19 taking turns with another tile's, 27 with seven),
         // the additions of the tile before in between.
         v4f t, before;
#pragma unroll
         for (int n = 0; n < TI * TJ; ++n) {
            const int i = n / TJ, j = n % TJ;
            constexpr int A[6] = {2, 1, 1, 0, 0, 0}, B[6] = {0, 0, 1, 1, 2, 0};
            t = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 6; ++m) {
               t = STORE == QUADS ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j][A[m]], w[i][B[m]], t, 0, 0, 0)
                                  : __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][B[m]], x[j][A[m]], t, 0, 0, 0);
               if (n > 0 && m >= 1 && m < 5) acc[(n - 1) / TJ][(n - 1) % TJ][m - 1] = __fadd_rn(acc[(n - 1) / TJ][(n - 1) % TJ][m - 1], before[m - 1]);
               __builtin_amdgcn_sched_barrier(0);
            }
            before = t;
            if (i == TI - 1) read_x(j, off);
            if (j + 1 == TJ) load_w(i, (unsigned)(step + 1));      // (behind the last step: read and not used)
            __builtin_amdgcn_sched_barrier(0);
         }
#pragma unroll
         for (int e = 0; e < 4; ++e) acc[TI - 1][TJ - 1][e] = __fadd_rn(acc[TI - 1][TJ - 1][e], before[e]);
      }
      if (!last) __syncthreads();
      if (more) {
#pragma unroll
         for (int s = 0; s < ITEMS; ++s)
            if (s * THREADS < items) put(xr, s, patch + (slot & 1) * g.slot_bytes);
      }
   }

   // (what was requested behind the last step is let in here: the compiler would wait for it between stores, and so for stores)
   __builtin_amdgcn_s_waitcnt(0);
   // sums that are not finite: again, tile by tile of 16 x 16, with fp32 instructions on the operands as they were given. One gathers 0.35 us for every four
   // products of a sum. us without one, with one infinity in x, one in every image, all sums above 2^95: 256x64x56x56 -> 128, 3x3 581 / 644 / 1190 / 13000;
   // 33x128x99x99 -> 128, 3x3 s2 171 / 550 / 624 / 4340 (1950 / 2050 / 5000 with all of a wavefront's tiles); 48x80x144x11 -> 192, 7x7 s2 171 / 1650 / 1760 / 4670;
   // transposed 64x128x28x28 -> 64, 4x4 s2 89 / 452 / 523 / 1890 (890 / 970 / 1830); 60x46x24x23 -> 64, 3x3 s2 31 / 92 / 104 / 336. The branch
   // lies behind the kernel: in front of the stores each of its instructions cost the others (two steps at a time 1.16 times longer at 13 us).
   v4f none = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
   for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
         for (int e = 0; e < 4; ++e) none[e] = fmaf(acc[i][j][e], 0.0f, none[e]);
   const float any = (none[0] + none[1]) + (none[2] + none[3]);
   unsigned again_of = 0;      // the tiles whose sums were formed again, a bit each
   int p1 = p0;      // (so that nothing of the pixels' places is kept in registers through the loop)
   asm volatile("" : "+s"(p1));
   if (__builtin_expect(__builtin_amdgcn_ballot_w64(any != 0.0f) != 0, 0)) {
      // (the arguments once more, from memory, and one tile after the other: in registers through the loop, for this branch, they cost 3 %
      // of every call and up to 13 with few channels. 32 channels x 128 pixels read the weights' alone again: with all of them the
      // compiler spills fragments in the loop.)
      constexpr bool ALL = (TI * TJ != 4 || WO == 1 || TI == 2);
      auto again = __builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(again));
      const SplitArgs &late = *(const SplitArgs *)again, &h = ALL ? late : g;
      const SplitPhase &weights = late.phase[PHASES || TOGETHER ? phase : 0], &f = ALL ? weights : q;
      const int ftaps = f.KH * f.KW;
      const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(h.x), 0, (int)h.xbytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(late.w0), 0, (int)OUTSIDE, 0x00020000);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
         for (int j = 0; j < TJ; ++j) {
            float z = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) z = fmaf(acc[i][j][e], 0.0f, z);
            if (__builtin_amdgcn_ballot_w64(z != 0.0f) != 0) again_of |= 1u << (i * TJ + j);
         }
      const int total = (h.icg + 3) / 4 * ftaps;
#pragma unroll 1
      for (unsigned left = again_of; left != 0; left &= left - 1) {
         const int tile = __builtin_ctz(left);
         const int p = p1 + (wp * TJ + tile % TJ) * 16 + r16, panel = fdiv(p, f.dPHW), r = p - panel * f.PHW, oy = fdiv(r, f.dWS), n = fdiv(panel, f.dStrips);
         const int iy0 = oy * h.sh + f.down - f.ph, ix0 = ((panel - n * f.strips) * f.ws + r - oy * f.ws) * h.sw + f.right - f.pw;
         const int oc = (tile0 + tile / TJ) * 16 + r16;
         v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
         int c = kg, t = 0;
         // (requests of two steps leave together)
#pragma unroll 1
         for (int step = 0; step < total; step += 2) {
            float xv[2], wv[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
               const int a = fdiv(t, f.dKW), b = t - a * f.KW, iy = iy0 + a * h.dh, ix = ix0 + b * h.dw;
               const bool in = p < f.P && r < f.full && c < h.icg && (unsigned)iy < (unsigned)h.H && (unsigned)ix < (unsigned)h.W;
               xv[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)(in ? (unsigned)(n * h.chw4 + (iy * h.W + ix) * 4 + (grp * h.icg + c) * h.hw4) : OUTSIDE), 0, 0));
               wv[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ors, (int)(c < h.icg && oc < h.ocg ? 4u * weight_at(late, weights, grp, oc, c, a, b, ROWS) : OUTSIDE), 0, 0));
               if (++t == ftaps) {
                  t = 0;
                  c += 4;
               }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
               if (step + u < total) sum = STORE == QUADS ? __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u], wv[u], sum, 0, 0, 0) : __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u], xv[u], sum, 0, 0, 0);
         }
#pragma unroll
         for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
               for (int e = 0; e < 4; ++e) acc[i][j][e] = tile == i * TJ + j ? sum[e] : acc[i][j][e];
      }
   }

   const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(g.y, 0, (int)g.ybytes, 0x00020000);
   const rsrc_t yrs4 = make_rsrc(g.y, g.ybytes);
   auto finish = [&](float v, float b, int tile) {
      v = __fmul_rn(v, again_of >> tile & 1 ? 1.0f : UNSCALE);
      if (g.bias) v = __fadd_rn(v, b);
      return g.relu ? (v > 0.0f ? v : 0.0f) : v;
   };
   // TOGETHER, two phases of neighbouring columns: each takes two of the other's four pixels and stores four columns next to each other
   v2f other[TOGETHER && STORE == QUADS ? TI : 1][TOGETHER && STORE == QUADS ? TJ : 1];
   if constexpr (TOGETHER && STORE == QUADS) {
      __syncthreads();      // the patch is read
      v2f *const swap = reinterpret_cast<v2f *>(smem_raw);
      const bool odd = q.ox0 != 0;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
         for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = finish(acc[i][j][e], bias[i][0], i * TJ + j);
            swap[((wave * TI + i) * TJ + j) * 64 + lane] = odd ? v2f{acc[i][j][0], acc[i][j][1]} : v2f{acc[i][j][2], acc[i][j][3]};
         }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
         for (int j = 0; j < TJ; ++j) other[i][j] = swap[(((wave ^ 1) * TI + i) * TJ + j) * 64 + lane];
   }
#pragma unroll
   for (int j = 0; j < TJ; ++j) {
      const int p = p1 + (wp * TJ + j) * 16 + (STORE == QUADS ? 4 * kg : r16);
      const int panel = fdiv(p, q.dPHW), r = p - panel * q.PHW, oy = fdiv(r, q.dWS), n = fdiv(panel, q.dStrips);
      const int ox = (panel - n * q.strips) * q.ws + r - oy * q.ws;
      const bool pixel = p < q.P && r < q.full && ox < q.OW && (!TOGETHER || oy < q.OH);
      const int column = TOGETHER && STORE == QUADS ? 2 * ox + 4 * q.ox0 : q.ox0 + ox * q.oxs;
      const unsigned at_pixel = (unsigned)(n * g.ocplane4 + ((q.oy0 + oy * q.oys) * g.OW0 + column) * 4);
#pragma unroll
      for (int i = 0; i < TI; ++i) {
         const int oc = (tile0 + i) * 16;
         if (oc >= g.ocg) continue;
         v4f v = acc[i][j];
         if constexpr (STORE == QUADS) {
            const bool there = pixel && oc + r16 < g.ocg;
            if constexpr (TOGETHER) {
               const v2f o = other[i][j];
               v = q.ox0 != 0 ? v4f{o[0], v[2], o[1], v[3]} : v4f{v[0], o[0], v[1], o[1]};
            } else {
#pragma unroll
               for (int e = 0; e < 4; ++e) v[e] = finish(v[e], bias[i][0], i * TJ + j);
            }
            store16_buf(yrs4, v, there ? at_pixel + (unsigned)(r16 * g.plane4) : OUTSIDE, (unsigned)(grp * g.ocg + oc) * (unsigned)g.plane4);
         } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
               if (oc + e >= g.ocg) continue;
               const bool there = pixel && oc + 4 * kg + e < g.ocg;
               __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, finish(v[e], bias[i][STORE == QUADS ? 0 : e], i * TJ + j)), yrs, (int)(there ? at_pixel + (unsigned)(kg * 4 * g.plane4) : OUTSIDE),
                                                     (int)((unsigned)(grp * g.ocg + oc + e) * (unsigned)g.plane4), 0);
            }
         }
      }
   }
}

struct SplitWeightArgs {
   const float *w;
   v4i *dst;
   int icg, ocg, octiles, KH0, KW0, transposed, rows, total;      // total: triples of 16-byte pieces over all phases
   SplitPhase phase[MAX_PHASES];
};

// The fragments [group][16 channels][step][h, m, l][lane][8 of K]; zeros behind the last channel and the last k.
__global__ void __launch_bounds__(256) k_conv_f32_split_weights(SplitWeightArgs g)
{
   const int idx = blockIdx.x * 256 + threadIdx.x;
   if (idx >= g.total) return;
   SplitPhase q = g.phase[0];
#pragma unroll
   for (int i = 1; i < MAX_PHASES; ++i)
      if (g.phase[i].wofs > 0 && 3 * idx >= g.phase[i].wofs) q = g.phase[i];
   int r = idx - q.wofs / 3;
   const int lane = r & 63;
   r >>= 6;
   const int step = r % q.steps, tile = r / q.steps;
   const int oc = (tile % g.octiles) * 16 + (lane & 15), grp = tile / g.octiles;
   const int chunk = 4 * step + (lane >> 4), c8 = fdiv(chunk, q.dTaps), t = chunk - c8 * q.KH * (g.rows ? 1 : q.KW);
   const int a = g.rows ? t : fdiv(t, q.dKW), b = t - a * q.KW;
   float v[8];
#pragma unroll
   for (int e = 0; e < 8; ++e) {
      const int ic = g.rows ? c8 : c8 * 8 + e;
      const bool in = oc < g.ocg && ic < g.icg && (!g.rows || e < q.KW);
      v[e] = in ? g.w[weight_at(g, q, grp, oc, ic, a, g.rows ? e : b, g.rows)] : 0.0f;
   }
   v4i s[3];
   split8(v, s);
   v4i *d = g.dst + q.wofs + ((size_t)tile * q.steps + step) * 192 + lane;
   d[0] = s[0];
   d[64] = s[1];
   d[128] = s[2];
}

template <int TI, int TJ>
int launch_together(sofie_hip_ctx *ctx, const SplitArgs &g, bool quads, long tiles)
{
   constexpr auto kern_p = k_conv_f32_split<TI, TJ, SplitPlan::TOGETHER, PIXELS, false, false>, kern_q = k_conv_f32_split<TI, TJ, SplitPlan::TOGETHER, QUADS, false, false>;
   SOFIE_LARGE_LDS(kern_p);
   SOFIE_LARGE_LDS(kern_q);
   const size_t patch = (size_t)(g.table_bytes + g.slot_bytes * (g.nslots > 1 ? 2 : 1)), swap = (size_t)4 * TI * TJ * 64 * 8;
   if (quads) hipLaunchKernelGGL(kern_q, dim3((unsigned)tiles), dim3(THREADS), patch > swap ? patch : swap, ctx->stream, g);
   else hipLaunchKernelGGL(kern_p, dim3((unsigned)tiles), dim3(THREADS), patch, ctx->stream, g);
   return check_launch(ctx, "k_conv_f32_split");
}

template <int TI, int TJ, int WO>
int launch(sofie_hip_ctx *ctx, const SplitArgs &g, int nphases, bool quads, bool rows, long tiles)
{
   auto start = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(tiles * nphases)), dim3(THREADS), (size_t)(g.table_bytes + g.slot_bytes * (g.nslots > 1 ? 2 : 1)), ctx->stream, g);
      return check_launch(ctx, "k_conv_f32_split");
   };
   if constexpr (TI * TJ <= 8 && TI <= 2) {
      constexpr auto rows_p = k_conv_f32_split<TI, TJ, WO, PIXELS, false, true>, rows_q = k_conv_f32_split<TI, TJ, WO, QUADS, false, true>;
      SOFIE_LARGE_LDS(rows_p);
      SOFIE_LARGE_LDS(rows_q);
      if (rows) return start(quads ? rows_q : rows_p);
   }
   constexpr auto kern_p = k_conv_f32_split<TI, TJ, WO, PIXELS, false, false>, kern_q = k_conv_f32_split<TI, TJ, WO, QUADS, false, false>,
                  kern_t = k_conv_f32_split<TI, TJ, WO, PIXELS, true, false>;
   SOFIE_LARGE_LDS(kern_p);
   SOFIE_LARGE_LDS(kern_q);
   SOFIE_LARGE_LDS(kern_t);
   return start(nphases > 1 ? kern_t : quads ? kern_q : kern_p);
}

// Few channels, a large kernel: a cell is the eight values that a row of the kernel meets at an output column, of one channel (a chunk of K:
// a row of the kernel, zeros up to eight), where that is 0.8 of the matrix cycles of the fp32 instructions or less: 5x5 and 7x7, not 3x3
// (three channels: 288 cycles for a tile of 16 x 16, 224 on the fp32 instructions).
bool rows_of(const ConvProblem &p, long icg)
{
   return icg < 6 && p.nphases == 1 && !p.transposed && p.KW0 <= 8 && 96 * ((icg * p.KH0 + 3) / 4) * 5 < 4 * 32 * ((icg * p.KH0 * p.KW0 + 3) / 4);
}

}  // namespace

int sofie::conv_f32_split(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done)
{
   *done = false;
   // The shortest form takes 6 us; below 7.5 us the choice among them costs the host more than it gives. Channels that fill little of the
   // chunks of eight, and short sums, which are their stores (60x1x16x72 -> 247, 3x3 27 us on k_conv_f32_any, 34 here; the tests of the
   // other kernels name them up to 144 products: 55x16x60x60 -> 64, 3x3, 1x10x101x101 -> 64).
   const long icg = p.C / p.groups;
   const bool rows = rows_of(p, icg);
   if (other_us < 7.5 + (ctx->constant_weights ? 0.0 : 4.0) || (!rows && icg < 6)) return SOFIE_HIP_OK;
   // (phases of short sums: all of them by one workgroup, with whole stores. 81x49x22x22 -> 47, 2x2 s2 33 us there with 4-byte stores, 28 on
   // k_conv_f32_any; 97x73x16x16 -> 27 13 and 17.5 with 16 bytes)
   ConvProblem united;
   const bool unites = SplitPlan::together(p, united);
   const bool brief = rows ? false : p.nphases == 1 ? icg * p.KH0 * p.KW0 <= 144 : icg * p.KH0 * p.KW0 < 48 * p.nphases;
   if (brief && !(unites && icg * p.KH0 * p.KW0 >= 64 && united.phase[0].OW % 4 == 0 && p.OW0 == 2 * united.phase[0].OW)) return SOFIE_HIP_OK;
   const size_t image = (size_t)p.C * p.H * p.W * 4, out_image = (size_t)p.OC * p.OH0 * p.OW0 * 4;
   // descriptors and OUTSIDE: 1 GiB of images per launch
   const size_t room = ((size_t)1 << 30) - ((size_t)16 << 20);
   if (image > room || out_image > room || p.nphases < 1 || p.nphases > MAX_PHASES) return SOFIE_HIP_OK;
   for (int i = 0; i < p.nphases; ++i) {
      const ConvPhase &f = p.phase[i];
      if (f.KH < 1 || f.KW < 1 || f.OH < 1 || f.OW < 1 || (long)f.KH * f.KW > 256) return SOFIE_HIP_OK;
   }
   SplitArgs g{};
   SplitPlan plan(p, rows);
   g.icg = plan.icg;
   g.ocg = plan.ocg;
   g.groups = p.groups;
   g.octiles = plan.octiles;
   size_t per = room / (image > out_image ? image : out_image);
   if (per > (size_t)p.N) per = (size_t)p.N;
   const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
   // (weights that are not kept are laid out in front of the launch, twice the bytes of k_conv_f32_any's)
   other_us = (other_us - (ctx->constant_weights ? 0.0 : 4.0)) * ((double)per / (double)p.N);
   SplitPlan::Form best{0, 0, 0, 0, 0, other_us};
   if (!brief) best = plan.choose(per, cus, other_us);
   const bool strided = !brief && p.nphases == 1 && (p.sh > 1 || p.sw > 1);
   if (strided) {
      // (slots of eight channels; estimates are off by some 8 %: 146x145x176x64 -> 40, 3x3 s2 529 us on k_conv_f32_any, 542 here)
      const SplitPlan::Form form = plan.choose_eights(per, cus, 0.95 * best.time);
      if (form.ti > 0) best = form;
   }
   SplitPlan one(unites ? united : p, false);
   if (unites) {
      // (k_conv_f32_any takes longer than its estimate under phases of unequal length: of 15 layers, 3x3 s2, this was the shorter way in all, by 1.07 to
      // 1.7 times; short sums stay there unless they are well ahead: 51x31x40x40 -> 185, 2x2 s2 88 us there, 92 here)
      const bool uneven = united.KH0 * united.KW0 % 4 != 0;
      const SplitPlan::Form form = one.choose_together(plan, per, cus, best.ti > 0 ? best.time : (uneven ? 1.2 : brief ? 0.85 : 1.0) * other_us);
      if (form.ti > 0) best = form;
   }
   if (best.ti == 0) return SOFIE_HIP_OK;
   auto prepare = [&] {
      const bool all = best.wo == SplitPlan::TOGETHER;
      g.CS = best.cs;
      g.nslots = plan.slots(best.cs);
      g.table_bytes = (all ? one : plan).table_bytes(best.cs);
      g.table_ints = all ? g.table_bytes / 16 : 0;
      g.slot_bytes = 0;
      for (int i = 0; i < p.nphases; ++i) {
         const ConvPhase &f = p.phase[i];
         SplitPhase &q = g.phase[i];
         SplitPlan::Panels s;
         if (all) one.panels(s, 0, best.pixels(), best.strips);
         else plan.panels(s, i, best.pixels(), best.strips);
         const ConvPhase &patch = all ? united.phase[0] : f;
         q.ws = s.ws; q.strips = s.strips; q.PHW = s.PHW; q.full = s.full;
         q.HP = s.HP; q.PW = s.PW; q.cells = s.cells;
         q.KH = f.KH; q.KW = f.KW; q.ph = patch.ph; q.pw = patch.pw;
         q.down = patch.ph - f.ph; q.right = patch.pw - f.pw;
         q.OH = f.OH; q.OW = f.OW;
         q.chunks = best.cs / 8 * plan.chunks[i];
         q.ring = (rows || q.chunks % 2 == 0 ? 2 : 4) * q.chunks;
         q.steps = plan.steps[i];
         q.wofs = (int)plan.wofs[i];
         q.oy0 = f.oy0; q.oys = f.oys; q.ox0 = f.ox0; q.oxs = f.oxs;
         q.th0 = f.th0; q.ths = f.ths; q.tw0 = f.tw0; q.tws = f.tws;
         if (SplitPlan::slot_bytes(q.cells, best.cs) > g.slot_bytes) g.slot_bytes = SplitPlan::slot_bytes(q.cells, best.cs);
         q.tiles = q.strips > 1 && q.PHW % best.pixels() == 0 ? q.PHW / best.pixels() : 0;
         q.dTiles = make_fastdiv((unsigned)(q.tiles > 0 ? q.strips * q.tiles : 1));
         q.dPHW = make_fastdiv((unsigned)q.PHW);
         q.dWS = make_fastdiv((unsigned)q.ws);
         q.dHP = make_fastdiv((unsigned)q.HP);
         q.dPW = make_fastdiv((unsigned)q.PW);
         q.dStrips = make_fastdiv((unsigned)q.strips);
         q.dTaps = make_fastdiv((unsigned)(q.KH * (rows ? 1 : q.KW)));
         q.dKW = make_fastdiv((unsigned)q.KW);
         q.dCells = make_fastdiv((unsigned)q.cells);
      }
      g.nphases = p.nphases;
      g.dPhases = make_fastdiv((unsigned)p.nphases);
      g.oblocks = cdiv(g.octiles, best.beside() * best.ti);
      g.dOB = make_fastdiv((unsigned)(g.oblocks * g.groups));
   };
   prepare();
   // the step behind the last one may be asked for, to no use
   const size_t wbytes = plan.pieces * 16 + 4096;
   g.wbytes = (unsigned)wbytes;
   int key[7 + 7 * MAX_PHASES] = {rows ? 6 : 5, p.groups, g.ocg, g.icg, p.KH0 * 4096 + p.KW0, p.transposed, p.nphases};
   for (int i = 0; i < p.nphases; ++i) {
      const SplitPhase &q = g.phase[i];
      const int v[7] = {q.KH, q.KW, q.th0, q.ths, q.tw0, q.tws, q.wofs};
      for (int e = 0; e < 7; ++e) key[7 + 7 * i + e] = v[e];
   }
   void *ws = nullptr;
   bool fresh = true;
   // (while a graph is recorded the scratch buffer may be too small: the caller has other ways)
   if (packed_weights(ctx, p.w, layout_key(key, 7 + 7 * p.nphases), wbytes, &ws, &fresh)) return SOFIE_HIP_OK;
   if (fresh) {
      SplitWeightArgs a{};
      a.w = p.w; a.dst = static_cast<v4i *>(ws);
      a.icg = g.icg; a.ocg = g.ocg; a.octiles = g.octiles;
      a.KH0 = p.KH0; a.KW0 = p.KW0; a.transposed = p.transposed; a.rows = rows; a.total = (int)(plan.pieces / 3);
      for (int i = 0; i < MAX_PHASES; ++i) a.phase[i] = g.phase[i];
      hipLaunchKernelGGL(k_conv_f32_split_weights, dim3((unsigned)cdiv(a.total, 256)), dim3(256), 0, ctx->stream, a);
      if (int rc = check_launch(ctx, "k_conv_f32_split_weights")) return rc;
   }
   g.w = static_cast<const v4i *>(ws);
   g.w0 = p.w;
   g.bias = p.bias;
   g.KH0 = p.KH0; g.KW0 = p.KW0; g.transposed = p.transposed;
   g.H = p.H; g.W = p.W; g.sh = p.sh; g.sw = p.sw; g.dh = p.dh; g.dw = p.dw; g.relu = p.relu;
   g.chw4 = (int)image;
   g.hw4 = p.H * p.W * 4;
   g.ocplane4 = (int)out_image;
   g.plane4 = p.OH0 * p.OW0 * 4;
   g.OW0 = p.OW0;
   const bool eights = best.cs == 8 && !rows;
   for (size_t n0 = 0; n0 < (size_t)p.N; n0 += per) {
      const size_t n = (size_t)p.N - n0 < per ? (size_t)p.N - n0 : per;
      if (n != per) {
         best = best.wo == SplitPlan::TOGETHER ? one.choose_together(plan, n, cus, HUGE_VAL) : eights ? plan.choose_eights(n, cus, HUGE_VAL) : plan.choose(n, cus, HUGE_VAL);
         prepare();
      }
      g.x = p.x + n0 * (image / 4);
      g.y = p.y + n0 * (out_image / 4);
      g.xbytes = (unsigned)(n * image);
      g.ybytes = (unsigned)(n * out_image);
      long tiles = 0;
      for (int i = 0; i < p.nphases; ++i) {
         SplitPhase &q = g.phase[i];
         q.panels = (int)n * q.strips;
         q.P = q.panels * q.PHW;
         const long t = (long)cdiv(q.P, best.pixels()) * g.oblocks * g.groups;
         if (t > tiles) tiles = t;
      }
      int rc = SOFIE_HIP_OK;
      switch (best.ti * 100 + best.tj * 10 + best.wo) {
#define SOFIE_FORM(i, j, o) case i * 100 + j * 10 + o: rc = launch<i, j, o>(ctx, g, p.nphases, plan.quads(g.phase[0].strips), rows, tiles); break
         SOFIE_FORM(4, 4, 2); SOFIE_FORM(3, 4, 2); SOFIE_FORM(2, 4, 2); SOFIE_FORM(4, 2, 2); SOFIE_FORM(2, 2, 2); SOFIE_FORM(1, 4, 2); SOFIE_FORM(1, 2, 2);
         SOFIE_FORM(1, 4, 1);
      case 444: rc = launch_together<4, 4>(ctx, g, one.pairs(), tiles); break;
      case 344: rc = launch_together<3, 4>(ctx, g, one.pairs(), tiles); break;
      case 244: rc = launch_together<2, 4>(ctx, g, one.pairs(), tiles); break;
      case 144: rc = launch_together<1, 4>(ctx, g, one.pairs(), tiles); break;
#undef SOFIE_FORM
      }
      if (rc) return rc;
   }
   *done = true;
   return SOFIE_HIP_OK;
}
