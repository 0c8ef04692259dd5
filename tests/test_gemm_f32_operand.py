"""The addresses k_gemm_f32 asks for (sofie_amd/csrc/gemm_f32_operand.h), worked out on the host by the header that the kernel
is compiled from: no request touches an element in front of an operand's first or behind its last one, and every element of a
step arrives where the kernel reads it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstddef>
#include <cstdio>
#include <vector>
#define __device__
#define __forceinline__ inline

namespace sofie {

// A request's dwords inside the descriptor are read, the others arrive as zeros (buffer loads check every dword).
struct rsrc_t {
   const float *base;
   unsigned bytes;
};
const float *const START = reinterpret_cast<const float *>(size_t(1) << 40);   // never dereferenced
long long last_element, too_far, lds[128 * 32];     // lds: the element that landed in a cell, -1 a zero, -2 nothing
int lane;

rsrc_t make_rsrc(const float *base, unsigned bytes) { return {base, bytes}; }
void dma(rsrc_t r, unsigned dst, int voff, int soff, int dwords)
{
   for (int d = 0; d < dwords; ++d) {
      const unsigned long long at = (unsigned long long)(unsigned)voff + (unsigned)soff + 4u * d;
      long long element = -1;
      if (at + 4 <= r.bytes) {
         element = (r.base - START) + (long long)(at / 4);
         if (element < 0 || element > last_element) ++too_far;
      }
      lds[dst / 4 + lane * dwords + d] = element;
   }
}
void dma16(rsrc_t r, unsigned dst, int voff, int soff) { dma(r, dst, voff, soff, 4); }
void dma4(rsrc_t r, unsigned dst, int voff, int soff) { dma(r, dst, voff, soff, 1); }

}  // namespace sofie

#include "gemm_f32_operand.h"

using namespace sofie;

// Every step of every tile of an operand of `count` rows (columns) and K, without checks where the kernel may leave them out.
template <bool KM, int ROWS>
int check(int count, int K, int pad)
{
   const int ld = (KM ? count : K) + pad, steps = (K + 31) / 32;
   last_element = KM ? (long long)(K - 1) * ld + count - 1 : (long long)(count - 1) * ld + K - 1;
   int bad = 0;
   for (int first = 0; first < count; first += ROWS) {
      std::vector<F32Operand<KM, ROWS>> lanes(256);
      for (int t = 0; t < 256; ++t) lanes[t].init(START, ld, first, count, K, t);
      const int whole = lanes[0].whole_steps();
      if (whole > steps || whole + 1 < K / 32) ++bad;
      for (int kt = 0; kt < steps + 3; ++kt)
         for (int unchecked = 0; unchecked < (kt < whole ? 2 : 1); ++unchecked) {
            for (auto &c : lds) c = -2;
            too_far = 0;
            for (int t = 0; t < 256; ++t) {
               lane = t & 63;
               if (unchecked) lanes[t].template request<true>(kt, 0, t >> 6);
               else lanes[t].template request<false>(kt, 0, t >> 6);
            }
            long long wrong = 0;
            for (int r = 0; r < ROWS; ++r)
               for (int k = 0; k < 32; ++k) {
                  // where F32Fragments reads it; rows behind the matrix may hold anything
                  const int cell = KM ? k * ROWS + (r + 16 * ((k >> 2) & 3)) % ROWS : r * 32 + (((k >> 2) ^ ((r >> 1) & 7)) << 2) + (k & 3);
                  const int gk = kt * 32 + k;
                  if (first + r >= count) continue;
                  const long long want = gk >= K ? -1 : KM ? (long long)gk * ld + first + r : (long long)(first + r) * ld + gk;
                  wrong += lds[cell] != want;
               }
            if (too_far || wrong) {
               if (!bad)
                  printf("%s ROWS %d count %d K %d ld %d: tile at %d, step %d%s: %lld elements outside, %lld cells wrong\n", KM ? "[K][rows]" : "[rows][K]",
                         ROWS, count, K, ld, first, kt, unchecked ? " (unchecked)" : "", too_far, wrong);
               ++bad;
            }
         }
   }
   return bad;
}

template <int ROWS> int check_all()
{
   int bad = 0;
   for (int K : {1, 2, 3, 5, 31, 32, 33, 34, 64, 96, 99, 160, 256, 1024})
      for (int count : {1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 66, 95, 97, 128, 129, 130, 131, 257, 1001})
         for (int pad : {0, 1, 3, 4}) {
            if ((long long)count * K > 150000 && !(count == 1001 && K == 1024 && pad == 0)) continue;
            bad += check<true, ROWS>(count, K, pad) + check<false, ROWS>(count, K, pad);
         }
   // the longest rows whose offsets fit 32 bits: a step's 32 rows, or a tile's
   const int longest_km = (1 << 24) - 1, longest = (int)((1ll << 31) / 4 / ROWS) - 1;
   for (int K : {31, 33, 64})
      for (int count : {31, 128, 130}) bad += check<true, ROWS>(count, K, longest_km - count) + check<false, ROWS>(count, K, longest - K);
   return bad;
}

int main() { return check_all<32>() + check_all<64>() + check_all<96>() + check_all<128>() ? 1 : 0; }
"""


def test_requests_stay_inside_the_operand(tmp_path):
    src, exe = tmp_path / "operand.cpp", tmp_path / "operand"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wno-unknown-pragmas", "-I" + os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=300)
    assert res.returncode == 0, res.stdout[-3000:]
