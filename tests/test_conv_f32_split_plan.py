"""How k_conv_f32_split chooses tiles, slots and strips (sofie_amd/csrc/conv_f32_split_plan.h), on the host: the same choice as a search that
leaves no form out, and few estimates on the way (each call makes them, in front of launches that may take 6 us). No tile of 128 channels x
64 pixels where stores are four bytes, which takes up to 1.8 times its estimate."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "conv_f32_split_plan.h"
using namespace sofie;

// every form and slot, no bound in front of the strips
static double search(SplitPlan &plan, size_t n, double other_us, int icg, int octiles)
{
   static const int forms[][3] = {{2, 4, 2}, {2, 2, 2}, {4, 4, 2}, {3, 4, 2}, {4, 2, 2}, {1, 4, 2}, {1, 2, 2}, {1, 4, 1}};
   double best = other_us;
   for (const auto &f : forms) {
      if ((plan.rows && f[0] > 2) || (f[0] > 1 && f[2] * (f[0] - 1) >= octiles)) continue;
      for (int cs = plan.rows ? 8 * icg : 16; cs <= (plan.rows ? 8 * icg : 32); cs *= 2) {
         SplitPlan::Form form{f[0], f[1], f[2], cs, 0, 0.0};
         double least = HUGE_VAL;
         for (int strips = 1; strips <= 16; ++strips) {
            SplitPlan::Panels q[4], kinds[4];
            int cells = 0;
            bool fits = true;
            for (int i = 0; i < plan.nphases; ++i) {
               fits = fits && plan.panels(q[i], i, form.pixels(), strips) && (plan.slots(cs) == 1 || cs / 8 * plan.chunks[i] >= 4);
               if (fits && q[i].cells > cells) cells = q[i].cells;
            }
            if (!fits || cells * (cs / 8) > SplitPlan::items_of(f[0], f[1], f[2], plan.rows) * SplitPlan::THREADS) continue;
            if (plan.table_bytes(cs) + (plan.slots(cs) > 1 ? 2 : 1) * SplitPlan::slot_bytes(cells, cs) > SplitPlan::MAX_LDS) continue;
            if ((double)n * q[0].strips * q[0].PHW > (double)(1 << 30)) continue;
            if (f[0] == 4 && f[1] == 2 && !plan.quads(q[0].strips)) continue;
            for (int k = 0; k < plan.kinds; ++k) kinds[k] = q[plan.kind[k]];
            const double time = plan.estimate(form, kinds, n, 256) * (strips > 1 ? 1.02 : 1.0);
            if (time < least) least = time, form.strips = strips;
            else if (strips > form.strips + 1) break;
         }
         if (least < best) best = least;
      }
   }
   return best;
}

int main()
{
   srand(7);
   auto pick = [](int lo, int hi) { return lo + rand() % (hi - lo + 1); };
   long layers = 0, taken = 0, estimates = 0, without = 0, most = 0;
   while (layers < 3000) {
      ConvProblem p{};
      const int kind = rand() % 4;      // convolution, few channels, transposed 4x4 and 3x3 of stride 2
      const int k = kind == 1 ? pick(4, 8) : kind == 2 ? 4 : kind == 3 ? 3 : 2 * pick(0, 3) + 1, s = kind >= 2 ? 2 : pick(1, 2), pad = (k - 1) / 2;
      p.N = 1 << pick(0, 8), p.C = kind == 1 ? pick(1, 5) : pick(6, 260), p.OC = pick(8, 260), p.groups = 1;
      p.H = pick(5, 150), p.W = rand() % 2 ? p.H : pick(5, 224);
      p.dh = p.dw = 1, p.KH0 = p.KW0 = k, p.transposed = kind >= 2, p.nphases = kind >= 2 ? 4 : 1;
      p.sh = p.sw = kind >= 2 ? 1 : s;
      p.OH0 = kind >= 2 ? s * (p.H - 1) + k - 2 * pad : (p.H + 2 * pad - k) / s + 1;
      p.OW0 = kind >= 2 ? s * (p.W - 1) + k - 2 * pad : (p.W + 2 * pad - k) / s + 1;
      if ((double)p.N * p.C * p.H * p.W > (1 << 27) || (double)p.N * p.OC * p.OH0 * p.OW0 > (1 << 27)) continue;
      for (int i = 0; i < p.nphases; ++i) {
         ConvPhase &f = p.phase[i];
         if (kind < 2) f = {p.OH0, p.OW0, k, k, pad, pad, 0, 1, 0, 1, 0, 1, 0, 1};
         else f = {(p.OH0 + 1 - i / 2) / 2, (p.OW0 + 1 - i % 2) / 2, k == 4 ? 2 : 1 + i / 2, k == 4 ? 2 : 1 + i % 2, 1 - i / 2, 1 - i % 2, 0, 2, 0, 2, i / 2, 2, i % 2, 2};
      }
      const bool rows = kind == 1;
      const double other = rand() % 2 ? HUGE_VAL : 7.5 + rand() % 40;
      SplitPlan plan(p, rows), all(p, rows);
      const SplitPlan::Form form = plan.choose(p.N, 256, other);
      const double best = search(all, p.N, other, p.C, plan.octiles);
      if (form.time != best) return printf("layer %ld: %.17g, searched %.17g\n", layers, form.time, best), 1;
      if (form.ti == 4 && form.tj == 2 && !plan.quads(form.strips)) return printf("layer %ld: 128 channels x 64 pixels with 4-byte stores\n", layers), 1;
      ++layers;
      taken += form.ti > 0;
      estimates += plan.evaluated;
      without += all.evaluated;      // (its end of a row of strips that only get longer is the same)
      most = plan.evaluated > most ? plan.evaluated : most;
   }
   printf("%ld %ld %ld %ld %ld\n", layers, taken, estimates, without, most);
}
"""


def test_the_choice_of_a_full_search_with_few_estimates(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    layers, taken, estimates, without, most = map(int, out.stdout.split())
    assert layers == 3000 and taken > 1000
    assert estimates <= 6 * layers and most <= 50 and without >= 4 * estimates, out.stdout


STRIDES = r"""
#include <cstdio>
#include <cstdlib>
#include "conv_f32_split_plan.h"
using namespace sofie;

// every form, slot and row of strips; apart: the plan of the four phases, nullptr for slots of eight channels of a strided layer
static double search(SplitPlan &plan, const SplitPlan *apart, size_t n, double other_us)
{
   double best = other_us;
   for (int ti = 1; ti <= 4; ++ti)
      for (int tj = 2; tj <= 4; tj += 2)
         for (int cs = apart ? 16 : 8; cs <= (apart ? 32 : 8); cs *= 2) {
            SplitPlan::Form form{ti, tj, apart ? SplitPlan::TOGETHER : 2, cs, 0, 0.0};
            if ((apart && tj == 2) || (!apart && ti == 3 && tj == 2) || (ti > 1 && form.beside() * (ti - 1) >= plan.octiles)) continue;
            bool fits = true, even = true;
            for (int i = 0; apart && i < 4; ++i) even = even && apart->chunks[i] == apart->chunks[0];
            for (int i = 0; apart && i < 4; ++i) {
               const int chunks = cs / 8 * apart->chunks[i];
               fits = fits && (plan.slots(cs) == 1 || (chunks >= 4 && (even || chunks % 4 == 0)));
            }
            if (!fits || (!apart && plan.chunks[0] < 4)) continue;
            double least = HUGE_VAL;
            for (int strips = 1; strips <= 16; ++strips) {
               SplitPlan::Panels q;
               if (!plan.panels(q, 0, form.pixels(), strips) || q.cells * (cs / 8) > SplitPlan::items_of(ti, tj, form.wo, false) * SplitPlan::THREADS) continue;
               if (apart && strips > 1 && q.ws < 8) continue;
               if (plan.table_bytes(cs) + (apart && plan.slots(cs) == 1 ? 1 : 2) * SplitPlan::slot_bytes(q.cells, cs) > SplitPlan::MAX_LDS) continue;
               if (!apart && ti == 4 && tj == 2 && !plan.quads(q.strips)) continue;
               const double time = plan.estimate(form, &q, n, 256) * (strips > 1 ? 1.02 : 1.0);
               if (time < least) least = time, form.strips = strips;
               else if (!apart && strips > form.strips + 1) break;
            }
            if (least < best) best = least;
         }
   return best;
}

int main()
{
   srand(9);
   auto pick = [](int lo, int hi) { return lo + rand() % (hi - lo + 1); };
   long layers = 0, taken[2] = {0, 0}, estimates = 0, without = 0;
   while (layers < 2000) {
      ConvProblem p{};
      const int k = pick(2, 5);
      const bool up = k < 5 && (k != 3 || rand() % 2);      // transposed, 2x2, 3x3 and 4x4 of stride 2, or 3x3 and 5x5 of stride 2
      const int pad = (k - 1) / 2;
      p.N = 1 << pick(0, 8), p.C = pick(16, 260), p.OC = pick(8, 260), p.groups = 1;
      p.H = pick(5, 80), p.W = rand() % 2 ? p.H : pick(5, 100);
      p.dh = p.dw = 1, p.KH0 = p.KW0 = k, p.transposed = up, p.nphases = up ? 4 : 1, p.sh = p.sw = up ? 1 : 2;
      p.OH0 = up ? 2 * (p.H - 1) + k - 2 * pad : (p.H + 2 * pad - k) / 2 + 1;
      p.OW0 = up ? 2 * (p.W - 1) + k - 2 * pad : (p.W + 2 * pad - k) / 2 + 1;
      if ((double)p.N * p.C * p.H * p.W > (1 << 27) || (double)p.N * p.OC * p.OH0 * p.OW0 > (1 << 27)) continue;
      for (int i = 0; i < p.nphases; ++i) {
         const int a = i / 2, b = i % 2, z = k != 2;
         if (!up) p.phase[i] = {p.OH0, p.OW0, k, k, pad, pad, 0, 1, 0, 1, 0, 1, 0, 1};
         else p.phase[i] = {(p.OH0 + 1 - a) / 2, (p.OW0 + 1 - b) / 2, k == 4 ? 2 : 1 + z * a, k == 4 ? 2 : 1 + z * b, z * (1 - a), z * (1 - b), 0, 2, 0, 2, a, 2, b, 2};
      }
      const double other = 7.5 + rand() % 200;
      ConvProblem u;
      if (up && !SplitPlan::together(p, u)) return printf("layer %ld: not together\n", layers), 1;
      SplitPlan apart(p, false), plan(up ? u : p, false);
      const SplitPlan::Form form = up ? plan.choose_together(apart, p.N, 256, other) : plan.choose_eights(p.N, 256, other);
      const long made = plan.evaluated;
      const double best = search(plan, up ? &apart : nullptr, p.N, other);
      if (form.time != best) return printf("layer %ld: %.17g, searched %.17g\n", layers, form.time, best), 1;
      ++layers;
      taken[up] += form.ti > 0;
      estimates += made;
      without += plan.evaluated - made;
   }
   printf("%ld %ld %ld %ld\n", taken[0], taken[1], estimates, without);
}
"""


def test_strided_and_transposed_layers_by_a_full_search(tmp_path):
    src, exe = tmp_path / "strides.cpp", tmp_path / "strides"
    src.write_text(STRIDES)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    strided, transposed, estimates, without = map(int, out.stdout.split())
    assert strided > 200 and transposed > 200 and 2 * estimates <= without, out.stdout


LINEAR = r"""
#include <cstdio>
#include "conv_f32_split_plan.h"
using namespace sofie;

// images of one tile of every form, all channels in one block
int main()
{
   static const int forms[][3] = {{2, 4, 2}, {2, 2, 2}, {4, 4, 2}, {3, 4, 2}, {4, 2, 2}, {1, 4, 2}, {1, 2, 2}};
   for (const auto &f : forms) {
      ConvProblem p{};
      const int w = f[1] == 4 ? 16 : 8;
      p.N = 1, p.C = 16, p.OC = 32 * f[0], p.groups = 1, p.H = 8, p.W = w, p.dh = p.dw = p.sh = p.sw = 1, p.KH0 = p.KW0 = 3, p.nphases = 1, p.OH0 = 8, p.OW0 = w;
      p.phase[0] = {8, w, 3, 3, 1, 1, 0, 1, 0, 1, 0, 1, 0, 1};
      SplitPlan plan(p, false);
      const SplitPlan::Form form{f[0], f[1], f[2], 16, 1, 0.0};
      SplitPlan::Panels q;
      if (!plan.panels(q, 0, form.pixels(), 1)) return printf("no panels\n"), 1;
      const int round = 256 * 12;      // two, three or four workgroups to a compute unit
      const double one = plan.estimate(form, &q, round, 256), two = plan.estimate(form, &q, 2 * round, 256) - one;
      for (int k = 3; k <= 64; ++k) {
         const double time = plan.estimate(form, &q, (size_t)k * round, 256);
         if (std::fabs(time - one - (k - 1) * two) > 1e-9 * time) return printf("%d%d%d: %d rounds %.6f us, one %.6f, another %.6f\n", f[0], f[1], f[2], k, time, one, two), 1;
      }
      printf("%.3f ", one);
   }
}
"""


def test_estimates_grow_with_whole_rounds(tmp_path):
    """As many workgroups again take as long again, whatever the form and from whichever time on: no form is preferred from a certain time on."""
    src, exe = tmp_path / "linear.cpp", tmp_path / "linear"
    src.write_text(LINEAR)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert len(out.stdout.split()) == 7


CHOICES = r"""
#include <cstdio>
#include "conv_f32_split_plan.h"
using namespace sofie;

// a line per layer: N C H W OC KH KW, strides, pads (top left bottom right), dilations, groups, transposed (stride 2, no dilation)
int main()
{
   int N, C, H, W, OC, KH, KW, sh, sw, t, l, b, r, dh, dw, groups, up;
   while (scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d %d", &N, &C, &H, &W, &OC, &KH, &KW, &sh, &sw, &t, &l, &b, &r, &dh, &dw, &groups, &up) == 17) {
      ConvProblem p{}, u;
      p.N = N, p.C = C, p.OC = OC, p.groups = groups, p.H = H, p.W = W, p.KH0 = KH, p.KW0 = KW, p.transposed = up, p.nphases = up ? 4 : 1;
      p.sh = up ? 1 : sh, p.sw = up ? 1 : sw, p.dh = up ? 1 : dh, p.dw = up ? 1 : dw;
      p.OH0 = up ? 2 * (H - 1) + KH - t - b : (H + t + b - (KH - 1) * dh - 1) / sh + 1;
      p.OW0 = up ? 2 * (W - 1) + KW - l - r : (W + l + r - (KW - 1) * dw - 1) / sw + 1;
      // phase q of an axis: taps t0, t0 + 2, .., of which the last one reads the first row
      auto axis = [](int q, int out, int k, int pad, int &o, int &taps, int &ph) {
         const int t0 = (q + pad) & 1;
         o = (out - q + 1) / 2, taps = (k - t0 + 1) / 2, ph = (t0 + 2 * (taps - 1) - q - pad) / 2;
      };
      for (int i = 0; i < p.nphases; ++i) {
         ConvPhase &f = p.phase[i];
         if (!up) f = {p.OH0, p.OW0, KH, KW, t, l, 0, 1, 0, 1, 0, 1, 0, 1};
         else {
            f = {0, 0, 0, 0, 0, 0, 0, 2, 0, 2, i / 2, 2, i % 2, 2};
            axis(i / 2, p.OH0, KH, t, f.OH, f.KH, f.ph);
            axis(i % 2, p.OW0, KW, l, f.OW, f.KW, f.pw);
         }
      }
      if (up && !SplitPlan::together(p, u)) return printf("not together\n"), 1;
      SplitPlan plan(p, false), one(up ? u : p, false);
      const SplitPlan::Form other = plan.choose(N, 256, HUGE_VAL), form = up ? one.choose_together(plan, N, 256, HUGE_VAL) : plan.choose_eights(N, 256, HUGE_VAL);
      printf("%d %.3f %d\n", form.ti > 0, other.ti > 0 ? form.time / other.time : 0.0, one.quads(form.strips));
   }
}
"""


def test_layers_of_the_gpu_tests_take_the_forms_they_are_for(tmp_path):
    """Slots of eight channels and phases by one workgroup are reported under the same name as the other forms. Of the plan's forms they have the
    shortest estimate (by more than 5 % for slots of eight) on the layers that test them: where the kernel runs at all, it runs in these. Both kinds of stores
    with and without groups."""
    pytest.importorskip("torch")
    from test_gpu_conv_f32_split import EIGHTS, TOGETHER
    lines = [(n, c, h, w, oc, kh, kw, *s, *pads, *d, groups, 0) for n, c, h, w, oc, kh, kw, s, pads, d, groups in EIGHTS]
    lines += [(n, c, h, w, oc, k, k, 2, 2, a, a, b, b, 1, 1, groups, 1) for n, c, h, w, oc, k, (a, b), groups in TOGETHER]
    src, exe = tmp_path / "choices.cpp", tmp_path / "choices"
    src.write_text(CHOICES)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, v)) for v in lines), capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    found = [line.split() for line in out.stdout.splitlines()]
    assert len(found) == len(lines)
    for shape, (taken, ratio, _) in zip(EIGHTS + TOGETHER, found):
        assert taken == "1" and float(ratio) < (0.95 if shape in EIGHTS else 1.0), (shape, ratio)
    assert {(s[-1], q) for s, (_, _, q) in zip(TOGETHER, found[len(EIGHTS):])} == {(1, "0"), (1, "1"), (2, "0"), (2, "1")}
