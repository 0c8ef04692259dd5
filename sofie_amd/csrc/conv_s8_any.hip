// int8 convolution of any channel counts, kernel sizes, strides and pads (one group, int8 output) on the matrix cores.
//
// Implicit GEMM on v_mfma_i32_16x16x64_i8: rows are output pixels, columns output channels, K = 16-byte chunks of the
// input. A lane's operand of a K-step (64 bytes) is one chunk of its pixel, loaded straight into registers at
// base(pixel) + offset(chunk); the offsets of all chunks stand in a small LDS table. Two forms of the input:
//   * in place (BOUNDS): channels-last, C a multiple of 16, 16-byte aligned. A chunk lies inside one tap; a chunk outside
//     the image is replaced by the zero-point.
//   * a copy in scratch memory, [N][H + pads][W + pads][Cp], Cp = C rounded up to whole dwords, pads filled with the
//     zero-point: written by k_qconv_any_input from channels-last int8, by k_qconv_any_planes from channel planes, int8 or the float
//     tensor that QuantizeLinear would read. One kernel row of a window is then KW * Cp contiguous bytes, which are cut into chunks
//     together (a 7x7 kernel on 3 channels: 14 chunks instead of 49), and no tap needs a bounds check.
// The weights are copied fragment by fragment ([16 channels][K-step][lane][16 bytes], zeros behind the last channel and the
// last tap), so that what an operand reads behind a row or a pixel is multiplied by 0 and a fragment is 1 KB in one piece.
//
// Bound. The vector cache hands a CU 64 bytes a cycle: an operand fragment of 1 KB costs 16 cycles of it, a matrix
// instruction 16 cycles of one of four SIMDs, so 64 pixels x 64 channels per wavefront with the weights in LDS balance the
// two. Measurements stand at the rule in qconv_any.
#include <math.h>

#include "conv_s8.h"
#include "gemm_tile.h"

using namespace sofie;

namespace {

struct AnyArgs {
   const int8_t *x;         // channels-last input or its padded copy
   const int8_t *w;         // fragments of the weights
   const int32_t *bias;
   const float *scale;
   int8_t *y;
   unsigned xbytes, wbytes; // sizes of x and w: loads behind them return 0
   int M, OC;               // output pixels (pooled ones with the fused pooling), output channels
   int OH, OW;              // extent of the pixel grid of M
   int H, W, C;             // BOUNDS: the image
   int img, row;            // bytes of an image and of a row
   int sh, sw, ph, pw;      // BOUNDS: pads; otherwise 0
   int pix;                 // bytes of a pixel
   int run16;               // 16-byte chunks of a kernel row
   int S, chunks;           // K-steps of 64 bytes, chunks of 16 bytes in them that carry weights
   int nob;                 // blocks of NB*16 channels
   int ntiles, per;         // pixel tiles, consecutive tiles of a workgroup
   int total;               // workgroups with work (the grid is rounded up to the XCDs)
   int nhwc_out, plane;
   unsigned fill;
   int zp, lo;
   FastDiv dOW, dOH, dRun, dC16, dPlane;
};

constexpr unsigned OUTSIDE = 0x80000000u;

// MB x NB tiles of 16 pixels x 16 channels per wavefront; NW wavefronts, groups of WK of them share their pixels and deal
// the K-steps among themselves; D fragments of every pixel tile in flight. POOL: the four pixel tiles are the positions of
// a 2x2 window with stride 2. BLDS: the weights of the workgroup's channels stay in LDS while it walks over its tiles.
// (At least two wavefronts to a SIMD where weights are in LDS: left to itself the compiler took more than 256 registers with the accumulators for four
// wavefronts on four tiles of channels, one to a SIMD: 121x16x32x32 -> 128, 5x5 27.9 -> 21 us, 16x70x59x31 -> 97, 3x3 pooled 27.7 -> 12. One tile of channels takes 120
// to 180 registers, two tiles 160 to 186, so that two to four wavefronts share a SIMD, three and four tiles 189 to 256, two.)
template <int MB, int NB, int NW, int WK, int D, bool BOUNDS, bool POOL, bool BLDS>
__global__ void __launch_bounds__(NW * 64, BLDS ? 2 : 1) k_qconv_any(AnyArgs a)
{
   static_assert(!POOL || MB == 4, "the four window positions are the four pixel tiles");
   static_assert(!BLDS || WK == 1, "the dealt K-steps read their weights from memory");
   constexpr int MBP = POOL ? 1 : MB;
   constexpr int TM = (NW / WK) * MBP * 16;
   constexpr int OCT = NB * 16;
   extern __shared__ __align__(16) unsigned char smem[];
   float *const s_scale = reinterpret_cast<float *>(smem);
   int *const s_bias = reinterpret_cast<int *>(s_scale + OCT);
   v2i *const tab = reinterpret_cast<v2i *>(s_bias + OCT);                         // [S * 4] offset, (row << 16 | column) of a chunk
   unsigned char *const big = reinterpret_cast<unsigned char *>(tab + a.S * 4);    // weights (BLDS) or partial sums (WK > 1)

   const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
   const int l16 = lane & 15, kg = lane >> 4;
   const int wp = wave / WK, wk = wave % WK;
   // workgroups of one XCD (every eighth) take neighbouring pixel tiles: the rows that two tiles share are in its L2
   const int idx = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
   if (idx >= a.total) return;
   const int ob = idx % a.nob;
   const int t0 = (idx / a.nob) * a.per, t1 = min(t0 + a.per, a.ntiles);
   const int n0 = ob * OCT;

   const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(a.x), 0, a.xbytes, 0x00020000);
   const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(a.w), 0, a.wbytes, 0x00020000);

   if constexpr (BLDS) {
      // the fragments of NB tiles are contiguous: a linear copy by LDS-DMA, 1 KB per wavefront and request
      const rsrc_t rs = make_rsrc(a.w, a.wbytes);
      const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)big;
      for (int f = wave; f < NB * a.S; f += NW) dma16(rs, lds0 + f * 1024, lane * 16, (ob * NB * a.S + f) * 1024);
   }
   const int s_per = (a.S + WK - 1) / WK;
   const int s0 = wk * s_per, s1 = min(s0 + s_per, a.S);
   // offset and (row << 16 | column) of a chunk; chunks behind the last kernel row carry zero weights: they read the first chunk again
   auto chunk = [&](int q) {
      const int kh = fdiv(q, a.dRun), r = q - kh * a.run16;
      const int kw = BOUNDS ? fdiv(r, a.dC16) : 0;
      return q < a.chunks ? v2i{kh * a.row + r * 16, kh << 16 | kw} : v2i{0, 0};
   };
   float scale = 0.0f;
   int bias = 0;
   if (tid < OCT && n0 + tid < a.OC) {
      scale = a.scale[n0 + tid];
      if (a.bias) bias = a.bias[n0 + tid];
   }
   auto tables = [&](bool offsets) {
      if (offsets)
         for (int q = tid; q < a.S * 4; q += NW * 64) tab[q] = chunk(q);
      if (tid < OCT) {
         s_scale[tid] = scale;
         s_bias[tid] = bias;
      }
   };
   if constexpr (BLDS) {
      tables(true);
      wait_vmcnt<0>();
      __syncthreads();
   }

   const float zpo = (float)(a.zp + 128), lof = (float)(a.lo + 128);

   // sums of a tile (POOL: of the four positions) -> requantised bytes of pixel m, channels n0 + 16 i + 4 kg ..
   auto finish = [&](const v4i *s, int i, int m) {
      const v4f sc = *reinterpret_cast<const v4f *>(s_scale + i * 16 + kg * 4);
      const v4i bi = *reinterpret_cast<const v4i *>(s_bias + i * 16 + kg * 4);
      unsigned pk = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
         int v = s[0][t];
         if constexpr (POOL) {   // the requantisation is monotonic: falling for a negative scale
            const int hi = max(max(s[0][t], s[1][t]), max(s[2][t], s[3][t])), lo = min(min(s[0][t], s[1][t]), min(s[2][t], s[3][t]));
            v = sc[t] < 0.0f ? lo : hi;
         }
         const float r = __fmul_rn(__int2float_rn(v + bi[t]), sc[t]);
         pk = __builtin_amdgcn_cvt_pk_u8_f32(fmaxf(__fadd_rn(rintf(r), zpo), lof), t, pk);
      }
      pk ^= 0x80808080u;
      const int oc = n0 + i * 16 + kg * 4;
      if (m >= a.M || oc >= a.OC) return;
      if (a.nhwc_out) {
         int8_t *const p = a.y + (size_t)m * a.OC + oc;
         if (oc + 4 <= a.OC) __builtin_memcpy(p, &pk, 4);
         else
            for (int t = 0; t < a.OC - oc; ++t) p[t] = (int8_t)(pk >> (8 * t));
      } else {
         const int n = fdiv(m, a.dPlane);
         int8_t *const p = a.y + ((size_t)n * a.OC + oc) * a.plane + (m - n * a.plane);
         for (int t = 0; t < min(4, a.OC - oc); ++t) p[(size_t)t * a.plane] = (int8_t)(pk >> (8 * t));
      }
   };

   for (int tile = t0; tile < t1; ++tile) {
      int base[MB], ih0[MB], iw0[MB];
#pragma unroll
      for (int j = 0; j < MB; ++j) {
         int m = tile * TM + (POOL ? wp * 16 : (wp * MB + j) * 16) + l16;
         m = m < a.M ? m : a.M - 1;
         const int R = fdiv(m, a.dOW), n = fdiv(R, a.dOH);
         int oh = R - n * a.OH, ow = m - R * a.OW;
         if constexpr (POOL) { oh = 2 * oh + (j >> 1); ow = 2 * ow + (j & 1); }
         ih0[j] = oh * a.sh - a.ph;
         iw0[j] = ow * a.sw - a.pw;
         base[j] = n * a.img + ih0[j] * a.row + iw0[j] * a.pix;
      }
      v4i acc[NB][MB];
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
         for (int j = 0; j < MB; ++j) acc[i][j] = v4i{0, 0, 0, 0};

      v4i fa[D][MB], fb[BLDS ? 1 : D][NB];
      int pad[D][MB];      // BOUNDS: the zero-point where the chunk lies outside the image (its load returns 0), else 0
      auto load = [&](int buf, int s, v2i e) {
#pragma unroll
         for (int j = 0; j < MB; ++j) {
            unsigned off = (unsigned)(base[j] + e[0]);
            if constexpr (BOUNDS) {
               const bool in = (unsigned)(ih0[j] + (e[1] >> 16)) < (unsigned)a.H & (unsigned)(iw0[j] + (e[1] & 0xffff)) < (unsigned)a.W;
               off = in ? off : OUTSIDE;
               pad[buf][j] = in ? 0 : (int)a.fill;
            }
            fa[buf][j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 0, 0));
         }
         if constexpr (!BLDS) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
               fb[buf][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wrs, lane * 16, ((ob * NB + i) * a.S + s) * 1024, 0));
         }
      };
      auto mma = [&](int buf, int s) {
         v4i b[NB];
#pragma unroll
         for (int i = 0; i < NB; ++i) {
            if constexpr (BLDS) b[i] = *reinterpret_cast<const v4i *>(big + (i * a.S + s) * 1024 + lane * 16);
            else b[i] = fb[buf][i];
         }
#pragma unroll
         for (int j = 0; j < MB; ++j) {
            v4i f = fa[buf][j];
            if constexpr (BOUNDS) {
#pragma unroll
               for (int t = 0; t < 4; ++t) f[t] |= pad[buf][j];
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[i], f, acc[i][j], 0, 0, 0);
         }
      };
      // Weights from memory (one tile): the first requests leave with chunks that the wavefront works out by itself, and only steps
      // behind them need the table, which is written while they travel. Behind the barrier of the table and the scales, 16x48x35x29 -> 80,
      // 3x3 s2 took 6.5 us instead of 6.15.
      if (s0 < s1) {
#pragma unroll
         for (int u = 0; u < D; ++u) {
            if (!BLDS && s0 + u >= s1) break;
            const int s = min(s0 + u, s1 - 1);
            load(u, s, BLDS ? tab[s * 4 + kg] : chunk(s * 4 + kg));
         }
      }
      if constexpr (!BLDS) {
         tables(s_per > D);
         if (WK == 1 || s_per > D) __syncthreads();
      }
      if (s0 < s1) {
         int s = s0;
         for (; s + D < s1; s += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
               mma(u, s + u);
               const int next = min(s + u + D, s1 - 1);
               load(u, next, tab[next * 4 + kg]);
            }
         }
#pragma unroll
         for (int u = 0; u < D; ++u)
            if (s + u < s1) mma(u, s + u);
      }
      const int m0 = tile * TM + wp * MBP * 16 + l16;
      if constexpr (WK == 1) {
#pragma unroll
         for (int i = 0; i < NB; ++i) {
            if constexpr (POOL) finish(acc[i], i, m0);
            else
#pragma unroll
               for (int j = 0; j < MB; ++j) finish(&acc[i][j], i, m0 + j * 16);
         }
      } else {
         // sums of the wavefronts that share these pixels, added by whichever of them owns the unit
         v4i *const part = reinterpret_cast<v4i *>(big) + (size_t)wp * WK * NB * MB * 64;
#pragma unroll
         for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j) part[((wk * NB + i) * MB + j) * 64 + lane] = acc[i][j];
         __syncthreads();
         constexpr int UNIT = POOL ? MB : 1;
         for (int u = wk; u < NB * MB / UNIT; u += WK) {
            v4i v[UNIT];
#pragma unroll
            for (int e = 0; e < UNIT; ++e) {
               v[e] = part[(u * UNIT + e) * 64 + lane];
#pragma unroll
               for (int k = 1; k < WK; ++k) v[e] += part[(k * NB * MB + u * UNIT + e) * 64 + lane];
            }
            if constexpr (POOL) finish(v, u, m0);
            else finish(v, u / MB, m0 + (u % MB) * 16);
         }
         if (tile + 1 < t1) __syncthreads();
      }
   }
}

// Weights in fragment order: one thread per 16 bytes, [channel tile][K-step][lane].
__global__ void __launch_bounds__(256) k_qconv_any_weights(const int8_t *w, v4i *dst, int total, int S, int run16, FastDiv dS, FastDiv dRun,
                                                           FastDiv dPix, int pix, int OC, int C, int KH, int KW, int ohwi)
{
   const int id = blockIdx.x * 256 + threadIdx.x;
   if (id >= total) return;
   const int lane = id & 63, fs = id >> 6;
   const int t = fdiv(fs, dS), s = fs - t * S;
   const int oc = t * 16 + (lane & 15), q = s * 4 + (lane >> 4);
   const int kh = fdiv(q, dRun), r0 = (q - kh * run16) * 16;
   int8_t v[16];
#pragma unroll
   for (int b = 0; b < 16; ++b) {
      const int r = r0 + b, kw = fdiv(r, dPix), c = r - kw * pix;
      const bool ok = oc < OC && kh < KH && kw < KW && c < C;
      const size_t off = !ok ? 0 : ohwi ? (((size_t)oc * KH + kh) * KW + kw) * C + c : (((size_t)oc * C + c) * KH + kh) * KW + kw;
      const int8_t e = w[off];
      v[b] = ok ? e : (int8_t)0;
   }
   v4i o;
   __builtin_memcpy(&o, v, 16);
   dst[id] = o;
}

// The padded copy of the input from channels-last int8: 16 bytes of the copy per thread. What lies behind a pixel's last channel meets zero
// weights: it is what follows in the tensor. WHOLE: pixels of the copy are whole 16 bytes. Bound: the chain of divisions (one per thread and
// extent) and memory. With a thread per dword
// and now, us of both launches: 192x131x51x51 -> 12, 3x3 s2 88 / 51; 128x33x80x80 -> 13, 5x5 58 / 50; 60 random layers 1.1 times shorter in the mean, with the
// forms below 1.16.
template <bool WHOLE>
__global__ void __launch_bounds__(256) k_qconv_any_input(QConvArgs g, v4i *dst, int total, int HP, int WP, int cd, FastDiv dcd, FastDiv dWP, FastDiv dHP)
{
   ask_for_arguments<sizeof(g) + 48>();
   const int id = blockIdx.x * 256 + threadIdx.x;
   if (id >= total) return;
   const int p = fdiv(4 * id, dcd), R = fdiv(p, dWP), n = fdiv(R, dHP);
   int k = 4 * id - p * cd, c = p - R * WP - g.pw, r = R - n * HP - g.ph;
   const size_t bytes = (size_t)g.N * g.H * g.W * g.C;
   size_t row = ((size_t)n * g.H + r) * g.W;      // (of a row that is there)
   // (the last bytes of the tensor by themselves)
   auto load4 = [&](size_t at) {
      unsigned v = 0;
      if (at + 4 <= bytes) __builtin_memcpy(&v, g.x + at, 4);
      else
#pragma unroll
         for (int b = 0; b < 4; ++b)
            if (at + b < bytes) v |= (unsigned)(uint8_t)g.x[at + b] << (8 * b);
      return (int)v;
   };
   const int fill = (int)(0x01010101u * (unsigned)(g.zpx & 0xff));
   v4i v = {fill, fill, fill, fill};
   if constexpr (WHOLE) {
      if ((unsigned)r < (unsigned)g.H && (unsigned)c < (unsigned)g.W) {
         const size_t at = (row + c) * g.C + 4 * k;
         if (at + 16 <= bytes) __builtin_memcpy(&v, g.x + at, 16);
         else
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = load4(at + 4 * u);
      }
   } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
         int e = fill;
         if ((unsigned)r < (unsigned)g.H && (unsigned)c < (unsigned)g.W) e = load4((row + c) * g.C + 4 * k);
         v[u] = e;
         if (++k == cd) {
            k = 0;
            if (++c == WP - g.pw) {
               c = -g.pw;
               if (++r == HP - g.ph) r = -g.ph, row += (size_t)(g.H - HP) * g.W;      // (the next image's first row)
               row += g.W;
            }
         }
      }
   }
   dst[id] = v;
}

// The same from planes, int8 (FLOAT: the float tensor, quantized): a dword, four channels of a pixel, per thread; channels that no pixel has are
// not asked for or divided. 176x1x146x146 -> 16, 3x3 s2 33.5 -> 28 us (with four pixels per thread the same, and 202 -> 208 where it is 16 more
// divisions one behind the other: 185x3x160x96 -> 55, 7x7).
template <bool FLOAT>
__global__ void __launch_bounds__(256) k_qconv_any_planes(QConvArgs g, unsigned *dst, int pixels, int HP, int WP, int cd, FastDiv dPixels, FastDiv dWP, FastDiv dHP)
{
   ask_for_arguments<sizeof(g) + 48>();
   const int id = blockIdx.x * 256 + threadIdx.x, k = fdiv(id, dPixels);
   if (k >= cd) return;
   const int p = id - k * pixels, R = fdiv(p, dWP), n = fdiv(R, dHP), c = p - R * WP - g.pw, r = R - n * HP - g.ph;
   const int left = g.C - 4 * k;      // channels of this dword and behind it (what is not there meets zero weights)
   const size_t plane = (size_t)g.H * g.W;
   unsigned v = 0x01010101u * (unsigned)(g.zpx & 0xff);
   if ((unsigned)r < (unsigned)g.H && (unsigned)c < (unsigned)g.W) {
      const size_t off = ((size_t)n * g.C + (left > 0 ? 4 * k : 0)) * plane + (size_t)r * g.W + c;
      float f[4] = {};
      int q[4] = {};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
         if (t > 0 && t >= g.C) continue;
         const size_t at = off + (t < left ? t : 0) * plane;
         if constexpr (FLOAT) f[t] = g.xf[at];
         else q[t] = g.x[at];
      }
      v = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
         if (t > 0 && t >= g.C) continue;
         if constexpr (FLOAT) {
            const float z = fminf(fmaxf(rintf(__fdiv_rn(f[t], g.xscale)), -1024.0f), 1024.0f);
            q[t] = min(127, max(-128, (int)z + g.zpx));
         }
         v |= t < left ? (unsigned)(q[t] & 0xff) << (8 * t) : 0u;
      }
   }
   dst[(size_t)p * cd + k] = v;
}

size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

// Sizes that the launch and the scratch memory are planned by.
struct Plan {
   bool ok, copy;         // copy: the input goes through the padded copy
   int pix, HP, WP, run16, S, nt;
   size_t xbytes, wbytes;
};

Plan plan(const QConvArgs &g)
{
   Plan p{};
   const bool pool = g.pool_kh != 0;
   if (g.groups != 1 || !g.scale) return p;
   if (pool && !(g.pool_kh == 2 && g.pool_kw == 2 && g.pool_sh == 2 && g.pool_sw == 2)) return p;
   p.copy = g.xf || !g.x_nhwc || g.C % 16 != 0 || !aligned16(g.x);
   p.HP = g.H + g.ph + g.pbh;
   p.WP = g.W + g.pw + g.pbw;
   // pixels of whole dwords; from 64 channels on of whole chunks, so that no operand load crosses a cache line
   p.pix = !p.copy ? g.C : g.C >= 64 ? (g.C + 15) & ~15 : (g.C + 3) & ~3;
   const long long run = (long long)g.KW * p.pix, chunks = (run + 15) / 16 * g.KH;
   if (chunks > 4096 || g.KH > 0x7fff || g.KW > 0xffff) return p;
   p.run16 = (int)((run + 15) / 16);
   p.S = (int)((chunks + 3) / 4);
   p.nt = cdiv(g.OC, 16);
   p.wbytes = (size_t)(p.nt + 3) * p.S * 1024;   // the last block of up to four channel tiles may hang over by three
   const size_t in = p.copy ? (size_t)g.N * p.HP * p.WP * p.pix : (size_t)g.N * g.H * g.W * g.C;
   // 64 bytes behind the copy: a kernel row's last chunk reads up to 15 bytes behind the last pixel
   p.xbytes = p.copy ? in + 64 : in;
   const long long rows = (long long)g.N * p.HP, M = (long long)g.N * g.PH * g.PW;
   p.ok = p.xbytes < ((size_t)1 << 30) && p.wbytes < ((size_t)1 << 30) && rows < (1ll << 31) && M < (1ll << 30) && g.OC < (1 << 24);
   return p;
}

}  // namespace

namespace sofie {

size_t qconv_any_scratch(const QConvArgs &g)
{
   const Plan p = plan(g);
   return !p.ok ? 0 : up256(p.copy ? p.xbytes : 0) + up256(p.wbytes);
}

// One thread per output is the shorter way for a layer of a few million multiply-adds on few channels: one launch, where this one
// has a copy of the weights in front of it (2.7 us, unless it is kept) and one of the input (2.8 us, unless it is read in place),
// but a chain of K loads. Both estimates are fits to 1714 layers of 1 to 256 channels (9 % rms for the single thread's; what is
// chosen is more than 10 % behind the other in 10 of them without kept weights and in 6 with them). us, one thread / this without
// and with kept weights: 8x9x11x11 -> 85, 1x1 4.8 / 10.6 / 8.4; 1x3x32x32 -> 16, 3x3 6.8 / 10.9 / 8.2; 2x12x16x16 -> 20, 3x3
// 16.1 / 11.0 / 8.3; 1x16x14x14 -> 32, 3x3 in place 20.2 / 8.0 / 5.4.
bool qconv_any_pays(const sofie_hip_ctx *ctx, const QConvArgs &g)
{
   const double K = (double)g.C * g.KH * g.KW, outputs = (double)g.N * g.OC * g.OH * g.OW;
   // (what is fused here is a pass of its own there)
   const double passes = (g.pool_kh != 0 ? 4.0 : 0.0) + (g.xf ? 4.0 : 0.0);
   const double plain = 4.0 + passes + (g.x_nhwc ? 0.076 : 0.111) * K + 0.08 * g.KH * g.KW + 0.26e-6 * outputs * K + 2.9e-6 * outputs;
   return plain >= 5.0 + (plan(g).copy ? 2.8 : 0.0) + (ctx->constant_weights ? 0.0 : 2.7);
}

int qconv_any(sofie_hip_ctx *ctx, const QConvArgs &g, int8_t *scratch, bool *done)
{
   *done = false;
   const Plan p = plan(g);
   if (!p.ok) return SOFIE_HIP_OK;
   const bool pool = g.pool_kh != 0;
   int8_t *const xs = scratch, *const ws_own = scratch + up256(p.copy ? p.xbytes : 0);
   // weights: kept under the constant-weights promise, otherwise (and where packed_weights has only the start of the scratch
   // buffer to give) in this call's part of the scratch buffer
   void *ws = nullptr;
   bool fresh = true;
   const int layout[] = {4, g.OC, g.C, g.KH, g.KW, p.pix, g.w_ohwi};
   if (ctx->constant_weights)
      if (int rc = packed_weights(ctx, g.w, layout_key(layout, 7), p.wbytes, &ws, &fresh)) return rc;
   if (!ws || ws == ctx->workspace) ws = ws_own;
   if (fresh) {
      const int total = (int)(p.wbytes / 16);
      hipLaunchKernelGGL(k_qconv_any_weights, dim3(cdiv(total, 256)), dim3(256), 0, ctx->stream, g.w, static_cast<v4i *>(ws), total, p.S,
                         p.run16, make_fastdiv(p.S), make_fastdiv(p.run16), make_fastdiv(p.pix), p.pix, g.OC, g.C, g.KH, g.KW, g.w_ohwi);
      if (int rc = check_launch(ctx, "k_qconv_any_weights")) return rc;
   }
   if (p.copy) {
      const int cd = p.pix / 4, pixels = g.N * p.HP * p.WP, total = cdiv(pixels * cd, 4);
      const FastDiv dcd = make_fastdiv(cd), dWP = make_fastdiv(p.WP), dHP = make_fastdiv(p.HP), dPixels = make_fastdiv(pixels);
      const dim3 block(256), grid((unsigned)cdiv(g.xf || !g.x_nhwc ? pixels * cd : total, 256));
      unsigned *const dst = reinterpret_cast<unsigned *>(xs);
      v4i *const dst4 = reinterpret_cast<v4i *>(xs);
      if (g.xf) hipLaunchKernelGGL(k_qconv_any_planes<true>, grid, block, 0, ctx->stream, g, dst, pixels, p.HP, p.WP, cd, dPixels, dWP, dHP);
      else if (!g.x_nhwc) hipLaunchKernelGGL(k_qconv_any_planes<false>, grid, block, 0, ctx->stream, g, dst, pixels, p.HP, p.WP, cd, dPixels, dWP, dHP);
      else if (cd % 4 == 0) hipLaunchKernelGGL(k_qconv_any_input<true>, grid, block, 0, ctx->stream, g, dst4, total, p.HP, p.WP, cd, dcd, dWP, dHP);
      else hipLaunchKernelGGL(k_qconv_any_input<false>, grid, block, 0, ctx->stream, g, dst4, total, p.HP, p.WP, cd, dcd, dWP, dHP);
      if (int rc = check_launch(ctx, g.xf || !g.x_nhwc ? "k_qconv_any_planes" : "k_qconv_any_input")) return rc;
   }
   AnyArgs a{};
   a.x = p.copy ? xs : g.x;
   a.w = static_cast<const int8_t *>(ws);
   a.bias = g.bias; a.scale = g.scale; a.y = static_cast<int8_t *>(g.y);
   a.xbytes = (unsigned)p.xbytes; a.wbytes = (unsigned)p.wbytes;
   a.OC = g.OC; a.OH = g.PH; a.OW = g.PW; a.M = g.N * g.PH * g.PW;
   a.H = g.H; a.W = g.W; a.C = g.C;
   a.pix = p.pix;
   a.row = (p.copy ? p.WP : g.W) * p.pix;
   a.img = (p.copy ? p.HP : g.H) * a.row;
   a.sh = g.sh; a.sw = g.sw;
   a.ph = p.copy ? 0 : g.ph; a.pw = p.copy ? 0 : g.pw;
   a.run16 = p.run16; a.S = p.S; a.chunks = p.run16 * g.KH;
   a.nhwc_out = g.y_nhwc; a.plane = g.PH * g.PW;
   a.fill = 0x01010101u * (unsigned)(g.zpx & 0xff);
   a.zp = g.zpy; a.lo = g.lo;
   a.dOW = make_fastdiv(a.OW); a.dOH = make_fastdiv(a.OH); a.dRun = make_fastdiv(p.run16); a.dC16 = make_fastdiv(cdiv(p.pix, 16));
   a.dPlane = make_fastdiv(a.plane);
   const bool bounds = !p.copy && (g.ph || g.pw || g.pbh || g.pbw);

   const int cus = ctx->num_cus;
   const size_t tab_bytes = (size_t)p.S * 32;
   auto go = [&](auto kern, int nb, int nw, int wk, int mbp, size_t big, int resident) {
      const int tm = nw / wk * mbp * 16;
      a.nob = cdiv(p.nt, nb);
      a.ntiles = cdiv(a.M, tm);
      a.per = 1;
      if (resident) {      // persistent: one round of workgroups
         int groups = cus * resident / a.nob;
         if (groups < 1) groups = 1;
         a.per = cdiv(a.ntiles, groups);
      }
      a.total = cdiv(a.ntiles, a.per) * a.nob;
      hipLaunchKernelGGL(kern, dim3((unsigned)((a.total + 7) & ~7)), dim3(nw * 64), (size_t)nb * 16 * 8 + tab_bytes + big, ctx->stream, a);
      *done = true;
      return check_launch(ctx, "k_qconv_any");
   };
#define SOFIE_ANY(MB_, MBPOOL_, NB_, NW_, WK_, D_, BLDS_, big_, resident_)                                                   \
   do {                                                                                                                      \
      constexpr auto kb = k_qconv_any<MB_, NB_, NW_, WK_, D_, true, false, BLDS_>, kn = k_qconv_any<MB_, NB_, NW_, WK_, D_, false, false, BLDS_>, \
                     pb = k_qconv_any<4, NB_, NW_, WK_, D_, true, true, BLDS_>, pn = k_qconv_any<4, NB_, NW_, WK_, D_, false, true, BLDS_>; \
      SOFIE_LARGE_LDS(kb); SOFIE_LARGE_LDS(kn); SOFIE_LARGE_LDS(pb); SOFIE_LARGE_LDS(pn);                                    \
      return go(pool ? (bounds ? pb : pn) : (bounds ? kb : kn), NB_, NW_, WK_, pool ? 1 : MB_, big_, resident_);             \
   } while (0)
   // The form, by the number of workgroups it gives and by what the LDS holds.
   //   A, B  64 pixels x up to 64 channels per wavefront, weights in LDS, as many workgroups as are resident at once walk over the
   //         tiles: for a tile per compute unit and more, with 16 KB of weights and more from half of that (unpooled ones from six K-steps on:
   //         3x32x96x152 -> 188, 3x3 s2 on five 6.8 us in C, 7.95 here; and where the LDS holds as many tiles of channels as a wavefront: else C, D or E
   //         0.80 to 1.26 times as long over seven, 56x155x13x13 -> 120, 5x5 pooled 17.4 in D, 22.9 here). Not where the LDS holds one tile of channels of several, each of which would
   //         read all of the input: C, D or E take 0.39 to 1.04 times as long there, 0.64 in the mean of 17 (46x128x8x8 -> 252, 7x7 pooled 23.0 us, 32.4
   //         here). A: four wavefronts, up to three workgroups in a compute unit; B: eight wavefronts, one workgroup, from four rounds of tiles on
   //         with up to 75 KB of weights: 0.94 times A's time in the mean of 161 layers (three and four tiles of channels 0.91, of which A holds two
   //         wavefronts to a SIMD as well), with more weights 1.095 over 17, with two to four rounds 1.05 over 90. Four K-steps and fewer of an unpooled copy
   //         stay in A, whose third wavefront to a SIMD covers the trips to memory: B 1.034 times as long over 60, 0.91 to 1.14 (192x3x181x192 -> 25, 5x5
   //         122 us in A, 139 in B).
   //   C, D, E  weights from memory, below.
   // Channels per workgroup: up to four tiles of 16, as few idle ones as possible.
   auto even = [&](int most) { return cdiv(p.nt, cdiv(p.nt, most)); };
   const int mb = pool ? 1 : 4;
   int nb = even(4);
   while (nb > 1 && (size_t)nb * p.S * 1024 > (size_t)144 * 1024) nb = even(nb - 1);
   const size_t wlds = (size_t)nb * p.S * 1024;
   const long long big_tiles = (long long)cdiv(a.M, 4 * mb * 16) * cdiv(p.nt, nb);
   const bool half = 2 * big_tiles >= cus && wlds >= (size_t)16 * 1024 && nb == even(4) && (pool || p.S >= 6);
   if ((big_tiles >= cus || half) && wlds <= (size_t)144 * 1024 && (nb > 1 || even(4) == 1)) {
      const bool few_steps = p.copy && !pool && nb <= 2 && p.S <= 4;
      if (big_tiles < 4 * cus || wlds + tab_bytes > (size_t)75 * 1024 || few_steps) {
         const int resident = (int)((size_t)156 * 1024 / (wlds + tab_bytes + 1024)) > 3 ? 3 : (int)((size_t)156 * 1024 / (wlds + tab_bytes + 1024));
         if (nb == 1) SOFIE_ANY(4, 4, 1, 4, 1, 4, true, wlds, resident);
         if (nb == 2) SOFIE_ANY(4, 4, 2, 4, 1, 4, true, wlds, resident);
         if (nb == 3) SOFIE_ANY(4, 4, 3, 4, 1, 3, true, wlds, resident);
         SOFIE_ANY(4, 4, 4, 4, 1, 3, true, wlds, resident);
      }
      if (nb == 1) SOFIE_ANY(4, 4, 1, 8, 1, 4, true, wlds, 1);
      if (nb == 2) SOFIE_ANY(4, 4, 2, 8, 1, 4, true, wlds, 1);
      if (nb == 3) SOFIE_ANY(4, 4, 3, 8, 1, 3, true, wlds, 1);
      SOFIE_ANY(4, 4, 4, 8, 1, 3, true, wlds, 1);
   }
   // Fewer tiles: weights from memory. C: 32 pixels (pooled 16) x up to four or two tiles of channels, a wavefront has all of K; else
   // the K-steps dealt to four wavefronts (D: 16 or 32 pixels x 32 channels, E: 16 x 16) or eight (E). Microseconds: a launch and
   // the requests one behind the other, and per workgroup of a compute unit its wavefronts' starts, operands (more by the ones requested
   // in vain behind a short K), sums and conversions. A fit to 457 random layers of 16 to 256 channels with kept weights, a third of them
   // pooled, on which the forms differ: what it picks is 1.7 % behind the best of ten forms in the mean and 1.14 times faster than
   // a rule by tiles alone with eight wavefronts in every dealt form (16x48x35x29 -> 80, 3x3 s2 6.2 -> 4.1 us; 14792 pooled pixels -> 48
   // on 7 K-steps 26.9 -> 6.3; 14x14x512 -> 512, 3x3 9.2 -> 6.3). Pooled and in place, with the bounds of four windows to look up, requests behind
   // the first ones take longer than in the fit where nothing else runs meanwhile: 14 of 384 layers with fewer tiles than half of the compute units go from four
   // wavefronts to eight by it, all of them faster, 1.05 to 1.15 times (38x64x8x8 -> 69, 7x7 9.2 -> 8.0, 72x192x13x13 -> 9, 3x3 7.45 -> 6.75; with five steps
   // for each of four 4x128x8x8 -> 48, 3x3 6.2 -> 5.7).
   struct Few {
      int mb, nb, nw, wk, d;
   };
   const Few few[] = {{2, even(4), 4, 1, even(4) == 1 ? 4 : 3}, {2, even(2), 4, 1, even(2) == 1 ? 4 : 3}, {1, 2, 4, 4, 4}, {2, 2, 4, 4, 4}, {1, 1, 4, 4, 4}, {1, 1, 8, 8, 4}};
   int pick = 0;
   float least = 1e30f;
   for (int f = 0; f < 6; ++f) {
      const Few &q = few[f];
      if (q.nb > p.nt) continue;      // tiles of nothing
      const float workgroups = (float)cdiv(a.M, q.nw / q.wk * (pool ? 1 : q.mb) * 16) * (float)cdiv(p.nt, q.nb), per_cu = workgroups > (float)cus ? workgroups / (float)cus : 1.0f;
      const int steps = cdiv(p.S, q.wk), mbs = pool ? 4 : q.mb, pieces = mbs * q.nb;
      const bool looked_up = pool && bounds && q.wk > 1 && workgroups <= (float)cus;
      const float first = looked_up ? 0.753f : 0.353f, others = looked_up ? 0.503f : 0.153f;
      const float waits = 2.681f + (q.wk > 1 ? 0.068f : 0.0f) + (steps > q.d ? first + others * (float)(steps - q.d) / (float)q.d : 0.0f);
      const float work = (float)q.nw * (0.0379f + ((float)steps + 0.211f * (float)q.d) * (0.0126f * (float)mbs + 0.0059f * (float)q.nb)) +
                         (0.022f * (float)(q.nw / q.wk) + (q.wk > 1 ? 0.0086f * (float)q.nw : 0.0f)) * (float)pieces;
      if (waits + per_cu * work < least) {
         least = waits + per_cu * work;
         pick = f;
      }
   }
   nb = few[pick].nb;
   const auto sums = [&](int waves, int m, int n) { return (size_t)waves * n * (pool ? 4 : m) * 1024; };
   if (pick == 2) SOFIE_ANY(1, 4, 2, 4, 4, 4, false, sums(4, 1, 2), 0);
   if (pick == 3) SOFIE_ANY(2, 4, 2, 4, 4, 4, false, sums(4, 2, 2), 0);
   if (pick == 4) SOFIE_ANY(1, 4, 1, 4, 4, 4, false, sums(4, 1, 1), 0);
   if (pick == 5) SOFIE_ANY(1, 4, 1, 8, 8, 4, false, sums(8, 1, 1), 0);
   if (nb == 1) SOFIE_ANY(2, 4, 1, 4, 1, 4, false, 0, 0);
   if (nb == 2) SOFIE_ANY(2, 4, 2, 4, 1, 3, false, 0, 0);
   if (nb == 3) SOFIE_ANY(2, 4, 3, 4, 1, 3, false, 0, 0);
   SOFIE_ANY(2, 4, 4, 4, 1, 3, false, 0, 0);
#undef SOFIE_ANY
}

}  // namespace sofie
