// fp32 NCHW convolutions whose outputs are sums of at most nine products (one channel under a 3x3 kernel, up to nine channels under a 1x1), on
// the vector unit: k_conv_f32_short.
//
// A sum this short is a few matrix instructions between the tables, operand loads, waits and stores of a tile. Here a lane owns two or
// four pixels, 64 apart in the row of all images' pixels, and keeps the K inputs of each in registers; the weights of an output channel are
// uniform, scalar loads; neighbouring lanes load and store neighbouring dwords, whatever the width of a row, and a channel is a
// uniform offset. (Four neighbouring pixels per lane and 16-byte stores: every load of a window touched 16 lines for 64 lanes,
// 256x1x40x40 -> 32, 3x3 27.6 us.)
//
// Bound: the stores (3.7 TB/s at 229x1x50x50 -> 170). us against k_conv_f32_any: 256x1x40x40 -> 32, 3x3 25.9 -> 15.0; 229x1x50x50 -> 170,
// 3x3 134 -> 106; 56x1x189x30 -> 33, 1x1 25.6 -> 10.5; random layers of at most nine products 1.1 to 2.7 times shorter, the same distance
// from 64 bits (3e-8 to 7e-8). Longer sums are bound by vector instructions, 2 K multiply-adds for 8 bytes: 16x12x129x129 -> 86, 1x1
// s2 17.7 -> 20.8, 11x16x51x167 -> 66, 1x1 18.6 -> 19.4; they stay.
#include "conv_f32.h"
#include "gemm_tile.h"

using namespace sofie;

namespace {

constexpr unsigned OUTSIDE = 0x40000000u;      // no descriptor of this file reaches it
constexpr int MAX_K = 9;

struct ShortArgs {
   const float *x, *w, *bias;
   float *y;
   unsigned xbytes, ybytes;
   int P, plane, H, W, OW, icg, ocg, sh, sw, ph, pw, relu;
   int ocb, oblocks;             // output channels of a workgroup, their blocks in a group
   int chw4, ocplane4, hw4;
   FastDiv dPlane, dRow, dOB;
   struct {
      int at, dy, dx;            // bytes from the window's first element, rows and columns of it
   } tap[MAX_K];
};

// THROUGH: stores written through the L2
template <int K, int PIXELS, bool THROUGH>
__global__ void __launch_bounds__(256) k_conv_f32_short(ShortArgs g)
{
   ask_for_arguments<sizeof(g)>();
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   const int grp = fdiv(blockIdx.y, g.dOB), oc0 = (blockIdx.y - grp * g.oblocks) * g.ocb;
   const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.x), 0, (int)g.xbytes, 0x00020000);
   const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(g.y, 0, (int)g.ybytes, 0x00020000);
   float x[PIXELS][K];
   unsigned at[PIXELS];
#pragma unroll
   for (int j = 0; j < PIXELS; ++j) {
      const int p = ((int)blockIdx.x * 4 + wave) * 64 * PIXELS + j * 64 + lane;
      const int n = fdiv(p, g.dPlane), r = p - n * g.plane, oy = fdiv(r, g.dRow), ox = r - oy * g.OW;
      const int iy = oy * g.sh - g.ph, ix = ox * g.sw - g.pw;
      const int first = n * g.chw4 + grp * g.icg * g.hw4 + (iy * g.W + ix) * 4;
      at[j] = p < g.P ? (unsigned)(n * g.ocplane4 + r * 4) : OUTSIDE;
#pragma unroll
      for (int t = 0; t < K; ++t) {
         const bool in = p < g.P && (unsigned)(iy + g.tap[t].dy) < (unsigned)g.H && (unsigned)(ix + g.tap[t].dx) < (unsigned)g.W;
         x[j][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, (int)(in ? (unsigned)(first + g.tap[t].at) : OUTSIDE), 0, 0));
      }
   }
   const int count = g.ocg - oc0 < g.ocb ? g.ocg - oc0 : g.ocb, oc1 = grp * g.ocg + oc0;
   const float *w = g.w + (size_t)oc1 * K;
   unsigned channel = (unsigned)oc1 * (unsigned)g.plane * 4u;
#pragma unroll 4
   for (int oc = 0; oc < count; ++oc) {
      float s[PIXELS] = {};
#pragma unroll
      for (int t = 0; t < K; ++t)
#pragma unroll
         for (int j = 0; j < PIXELS; ++j) s[j] = fmaf(w[t], x[j][t], s[j]);
      w += K;
      const float b = g.bias ? g.bias[oc1 + oc] : 0.0f;
#pragma unroll
      for (int j = 0; j < PIXELS; ++j) {
         if (g.bias) s[j] = __fadd_rn(s[j], b);
         if (g.relu) s[j] = s[j] > 0.0f ? s[j] : 0.0f;
         __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, s[j]), yrs, (int)at[j], (int)channel, THROUGH ? 17 : 0);      // sc0 sc1
      }
      channel += (unsigned)g.plane * 4u;
   }
}

template <int K>
int launch(sofie_hip_ctx *ctx, const ShortArgs &g, int k, int pixels, bool through, dim3 grid)
{
   if constexpr (K > 1)
      if (k < K) return launch<K - 1>(ctx, g, k, pixels, through, grid);
   const auto kern = pixels == 4 ? (through ? k_conv_f32_short<K, 4, true> : k_conv_f32_short<K, 4, false>) : (through ? k_conv_f32_short<K, 2, true> : k_conv_f32_short<K, 2, false>);
   hipLaunchKernelGGL(kern, grid, dim3(256), 0, ctx->stream, g);
   return check_launch(ctx, "k_conv_f32_short");
}

}  // namespace

int sofie::conv_f32_short(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done)
{
   *done = false;
   const int icg = p.C / p.groups, ocg = p.OC / p.groups;
   const ConvPhase &f = p.phase[0];
   // calls below 7.5 us are a launch's latency on every kernel
   if (other_us < 7.5 || p.nphases != 1 || p.transposed || (long)icg * p.KH0 * p.KW0 > MAX_K || ocg < 4) return SOFIE_HIP_OK;
   if (f.oys != 1 || f.oxs != 1 || f.oy0 != 0 || f.ox0 != 0 || f.OW != p.OW0 || f.OH != p.OH0) return SOFIE_HIP_OK;
   // descriptors and OUTSIDE: 1 GiB of images per launch; offsets of taps
   const size_t image = (size_t)p.C * p.H * p.W * 4, out_image = (size_t)p.OC * p.OH0 * p.OW0 * 4, room = (size_t)1 << 30;
   if (image > room || out_image > room || ((long)icg * p.H + (long)p.KH0 * p.dh) * p.W + (long)p.KW0 * p.dw >= (1l << 28)) return SOFIE_HIP_OK;
   const int k = icg * p.KH0 * p.KW0;
   const long per = (long)(room / (image > out_image ? image : out_image)), plane = (long)f.OH * f.OW;
   const long n_launch = per < p.N ? per : p.N;
   ShortArgs g{};
   // (weights and addresses are shared by twice the outputs: with both 256x1x40x40 -> 32, 3x3 17.9 -> 15.0 us; four on fewer pixels 58x1x22x22 -> 58, 3x3
   // 7.4 -> 10.6.) Four pixels per lane where eight channels at a time leave six workgroups for a compute unit, else two
   const int pixels = cdiv((int)(n_launch * plane), 1024) * p.groups * (long)cdiv(ocg, 8) >= 6l * ctx->num_cus ? 4 : 2;
   // written through the L2s where a store is whole 64-byte pieces and the end of the kernel would be their write-back: 139x1x9x64 -> 48, 3x3 (15 MB) 9.4 -> 8.8,
   // 16x1x62x56 -> 34, 1x1 (7.6 MB) 4.9 -> 5.6; planes of other sizes 133x1x130x130 -> 60, 3x3 162 -> 262
   const bool through = plane % 16 == 0 && out_image * p.N >= ((size_t)14 << 20) && (reinterpret_cast<uintptr_t>(p.y) & 63u) == 0;
   const long blocks = cdiv((int)(n_launch * plane), 256 * pixels);
   g.ocb = 64;
   while (g.ocb > 8 && blocks * p.groups * cdiv(ocg, g.ocb) < 6l * ctx->num_cus) g.ocb /= 2;
   g.oblocks = cdiv(ocg, g.ocb);
   if ((long)p.groups * g.oblocks > 65535) return SOFIE_HIP_OK;
   // outputs at 4 TB/s; vector instructions of a wavefront, four cycles each: the window's, and per channel its multiply-adds and stores
   const double bytes = 4.0 * plane * p.N * p.OC / 4e6;
   const double waves = (double)plane * p.N / 128.0;
   const double valu = waves * (p.groups * g.oblocks * (40.0 + 16.0 * k) + p.OC * (2.0 * k + 10.0)) * 4.0 / (4.0 * ctx->num_cus) / 2100.0;
   const double us = 3.0 + (bytes > valu ? bytes + 0.3 * valu : valu + 0.3 * bytes);
   if (us >= other_us) return SOFIE_HIP_OK;
   g.w = p.w; g.bias = p.bias;
   g.plane = (int)plane; g.H = p.H; g.W = p.W; g.OW = f.OW;
   g.icg = icg; g.ocg = ocg; g.sh = p.sh; g.sw = p.sw; g.ph = f.ph; g.pw = f.pw; g.relu = p.relu;
   g.chw4 = (int)image; g.ocplane4 = (int)out_image; g.hw4 = p.H * p.W * 4;
   g.dPlane = make_fastdiv((unsigned)plane);
   g.dRow = make_fastdiv((unsigned)f.OW);
   g.dOB = make_fastdiv((unsigned)g.oblocks);
   for (int t = 0; t < k; ++t) {
      const int c = t / (p.KH0 * p.KW0), a = t / p.KW0 % p.KH0, b = t % p.KW0;
      g.tap[t] = {((c * p.H + a * p.dh) * p.W + b * p.dw) * 4, a * p.dh, b * p.dw};
   }
   for (long n0 = 0; n0 < p.N; n0 += n_launch) {
      const long n = p.N - n0 < n_launch ? p.N - n0 : n_launch;
      g.x = p.x + (size_t)n0 * (image / 4);
      g.y = p.y + (size_t)n0 * (out_image / 4);
      g.xbytes = (unsigned)(n * image);
      g.ybytes = (unsigned)(n * out_image);
      g.P = (int)(n * plane);
      if (int rc = launch<MAX_K>(ctx, g, k, pixels, through, dim3((unsigned)cdiv(g.P, 256 * pixels), (unsigned)(p.groups * g.oblocks)))) return rc;
   }
   *done = true;
   return SOFIE_HIP_OK;
}
