// k_conv_f32_split (conv_f32_split.hip): tiles, slots of channels and strips for a layer, by an estimate of the time. The arithmetic
// alone, also for a host program that checks it against a search through everything.
//
// Every call works this out anew, in front of a launch that may take 6 us: forms (tile and slot) come in the order of what they take at
// least, by a bound on the cells that any strips need; those that cannot be shorter than the best so far are left before their strips are
// looked at, and what strips of an image need depends on the tile's pixels alone and is worked out once for all forms and for phases of the
// same sizes. us of a call on the host without its launches, every form laid out for up to 16 strips / now / without this kernel (2.7 GHz):
// 256x64x56x56 -> 128, 3x3 6.4 / 2.4 / 0.7; 1x128x56x56 -> 128, 3x3, which k_conv_f32_any takes, 5.9 / 1.3 / 0.7; transposed 1x111x25x25 -> 192,
// 4x4 s2, taken by it, too, 26 / 2.8 / 1.2, and 17.6 us a call on the device for 11.0 of the kernel; 300 random layers 1.5 / 0.73 / 0.50 in the
// mean, 17 / 3.2 / 1.3 at most. Slots of 8 channels add 0.55 to strided layers (2000 random ones, with the transposed), the form with a phase per
// wavefront 0.53 to transposed ones (2.6 without the bound, with the strips laid out for each form again; 10.3 and 3.6 at most).
#pragma once
#include <cmath>

#include "conv_f32_patch.h"
#include "conv_f32_problem.h"

namespace sofie {

struct SplitPlan {
   static constexpr int MAX_PHASES = 4;
   static constexpr int CELL = 48;            // LDS bytes of 8 channels of a cell: h, m, l
   static constexpr int THREADS = 256;
   static constexpr int MAX_STRIPS = 16;
   static constexpr long MAX_LDS = 160 * 1024;

   // Cells x 8 channels of a slot that a thread carries, at most: registers, which decide how many workgroups share a compute unit.
   // (Rows of a kernel as cells: one slot, whose registers are free again in front of the loop.)
   static constexpr int items_of(int ti, int tj, int wo, bool rows) { return rows || wo == 1 ? 4 : ti * tj > 8 ? 3 : 2; }
   // Workgroups a compute unit holds at once, by registers.
   static constexpr int resident_of(int ti, int tj, int wo) { return ti * tj > 8 ? 2 : ti * tj > 4 || wo == 1 ? 3 : 4; }

   // 16 wo ti channels x 64 / wo tj pixels per workgroup, slots of cs channels, an image in strips; rows: a row of the kernel as a cell.
   // wo = TOGETHER: a wavefront for each of four phases, 16 ti channels x 16 tj places of them.
   static constexpr int TOGETHER = 4;
   struct Form {
      int ti, tj, wo, cs, strips;
      double time;
      int pixels() const { return 64 / wo * tj; }
      int beside() const { return wo == TOGETHER ? 1 : wo; }      // wavefronts side by side along the channels
   };

   // Panels (strips of images) of one phase under tiles of some pixels
   struct Panels {
      int ws, strips;         // columns of a strip, strips of an image
      int PHW, full;          // pixels of a panel, up to whole tiles where tiles do not run on into the next; those that exist
      int HP, PW, cells;      // rows of a panel's input, cells of a row, of a tile's patch
   };

   // of the layer
   int icg, ocg, octiles, nphases;
   bool rows, whole;          // whole: pixels next to each other are stored next to each other
   bool one_for_all = false;     // one workgroup for all phases
   int steps[MAX_PHASES];     // of four chunks of eight, all of K
   int chunks[MAX_PHASES];    // of eight channels of a slot
   size_t wofs[MAX_PHASES], pieces;      // first 16-byte piece of a phase's fragments; all of them
   int kinds, kind[MAX_PHASES], count[MAX_PHASES];      // phases of the same sizes (all four of a 4x4 kernel of stride 2): the first of each kind, how many

   long evaluated = 0;        // estimates made, for the test

   SplitPlan(const ConvProblem &p, bool rows_) : rows(rows_), p(p)
   {
      icg = p.C / p.groups;
      ocg = p.OC / p.groups;
      octiles = (ocg + 15) / 16;
      nphases = p.nphases;
      const ConvPhase &f0 = p.phase[0];
      whole = nphases == 1 && f0.oys == 1 && f0.oxs == 1 && f0.oy0 == 0 && f0.ox0 == 0 && f0.OW == p.OW0 && f0.OH == p.OH0;
      pieces = 0;
      kinds = 0;
      for (int i = 0; i < nphases; ++i) {
         const ConvPhase &f = p.phase[i];
         int k = 0;
         while (k < kinds && !(p.phase[kind[k]].OH == f.OH && p.phase[kind[k]].OW == f.OW && p.phase[kind[k]].KH == f.KH && p.phase[kind[k]].KW == f.KW)) ++k;
         if (k == kinds) {
            kind[kinds] = i;
            count[kinds++] = 0;
         }
         ++count[k];
         chunks[i] = p.phase[i].KH * (rows ? 1 : p.phase[i].KW);
         steps[i] = ((rows ? icg : (icg + 7) / 8) * chunks[i] + 3) / 4;
         wofs[i] = pieces;
         pieces += (size_t)p.groups * octiles * steps[i] * 192;
      }
      for (Strips &s : strips_seen) s.seen = 0;
   }

   // Whether four pixels are stored at once.
   bool quads(int strips) const { return one_for_all ? pairs() : whole && (strips == 1 ? (long)p.OH0 * p.OW0 % 4 == 0 : p.OW0 % 4 == 0); }

   // Strips of phase i for tiles of bp pixels; false where numbers leave their range.
   bool panels(Panels &q, int i, int bp, int strips) const
   {
      const ConvPhase &f = p.phase[i];
      q.ws = (f.OW + strips - 1) / strips;
      if (f.OW % 4 == 0) q.ws = (q.ws + 3) & ~3;
      q.strips = (f.OW + q.ws - 1) / q.ws;
      const long full = (long)f.OH * q.ws;
      const long HP = (long)(f.OH - 1) * p.sh + (long)(f.KH - 1) * p.dh + 1, PW = rows ? q.ws : (long)(q.ws - 1) * p.sw + (long)(f.KW - 1) * p.dw + 1;
      if (full > (1 << 28) || HP > (1 << 28) || PW > 4096) return false;
      // tiles that do not run on into the next panel read fewer rows: where the last one is nearly full
      const int up = ((int)full + bp - 1) / bp * bp;
      const bool apart = (long)up * 100 <= full * 104;
      const long pixels = apart ? up : full;
      const long cells = split_patch_rows(bp, q.ws, pixels, f.OH, p.sh, f.KH, p.dh, apart) * PW;
      if (pixels > (1 << 28) || cells > 4 * THREADS) return false;
      q.full = (int)full;
      q.PHW = (int)pixels;
      q.HP = (int)HP;
      q.PW = (int)PW;
      q.cells = (int)cells;
      return true;
   }

   int slots(int cs) const { return (icg + cs - 1) / cs; }
   int table_bytes(int cs) const
   {
      int most = 0;
      for (int i = 0; i < nphases; ++i) most = chunks[i] > most ? chunks[i] : most;
      return (2 * (cs > 8 ? cs / 8 : 2) * most * 4 + 255) & ~255;      // (8 channels: four slots, whose chunks are whole steps)
   }
   // Cells a workgroup of this form can hold, by what its threads carry.
   int cells_of(const Form &f) const { return items_of(f.ti, f.tj, f.wo, rows) * THREADS / (f.cs / 8); }
   static int slot_bytes(int cells, int cs) { return cells * (cs / 8) * CELL; }

   // The form with the shortest estimate for n images on cus compute units, below other_us; ti = 0 where there is none.
   Form choose(size_t n, int cus, double other_us)
   {
      static const int forms[][3] = {{2, 4, 2}, {2, 2, 2}, {4, 4, 2}, {3, 4, 2}, {4, 2, 2}, {1, 4, 2}, {1, 2, 2}, {1, 4, 1}};
      Form best{0, 0, 0, 0, 0, other_us};
      if (pieces * 16 > ((size_t)1 << 29)) return best;
      for (int k = 0; k < kinds; ++k)
         for (int t = 0; t < 3; ++t) least_cells[t][k] = cells_at_least(p.phase[kind[k]], 64 << t);
      // what may be the shortest first
      struct Candidate {
         Form form;
         int order;
      } candidates[16];
      int count = 0;
      for (const auto &f : forms) {
         if (rows && f[0] > 2) continue;
         if (f[0] > 1 && f[2] * (f[0] - 1) >= octiles) continue;      // tiles of nothing
         for (int cs = rows ? 8 * icg : 16; cs <= (rows ? 8 * icg : 32); cs *= 2) {
            Form form{f[0], f[1], f[2], cs, 0, 0.0};
            // (a step reaches into one slot behind its first chunk's)
            bool enough = true;
            for (int k = 0; k < kinds; ++k) enough = enough && least_cells[tile_of(form)][k] <= cells_of(form) && (slots(cs) == 1 || cs / 8 * chunks[kind[k]] >= 4);
            if (!enough) continue;
            form.time = least_time(form, n, cus);
            if (form.time >= best.time) continue;
            int at = count++;
            for (; at > 0 && candidates[at - 1].form.time > form.time; --at) candidates[at] = candidates[at - 1];
            candidates[at] = {form, (int)(&f - forms) * 2 + (cs == 32)};
         }
      }
      int order = 16;
      for (int c = 0; c < count && candidates[c].form.time <= best.time; ++c) {
         Form form = candidates[c].form;
         form.time = HUGE_VAL;
         const int cs = form.cs, bp = form.pixels(), room = cells_of(form);
         Strips &s = strips_seen[tile_of(form)];
         // (as many strips as the estimate says: fewer cells for a tile's pixels against whole lines per store, 4-byte stores where strips are no
         // whole fours, 256x64x10x10 -> 128 29.5 us in one strip, 36.2 in five of two columns; by the number of cells alone 42x59x79x62 -> 9, 3x3 66.5,
         // now 44.5, and k_conv_f32_any 58.7)
         for (int strips = 1; strips <= MAX_STRIPS; ++strips) {
            if (strips > s.seen) look_at(s, bp, strips);
            const Panels *q = s.panels[strips - 1];
            if (s.cells[strips - 1] == 0 || s.cells[strips - 1] > room) continue;
            if (table_bytes(cs) + (slots(cs) > 1 ? 2 : 1) * (long)slot_bytes(s.cells[strips - 1], cs) > MAX_LDS) continue;
            if ((double)n * q[0].strips * q[0].PHW > (double)(1 << 30)) continue;
            // (128 channels x 64 pixels with 4-byte stores take up to 1.8 times what the estimate says, and more than the next form: transposed
            // 23x110x51x10 -> 256, 3x3 s2 108 us, 64 without it, 83 on k_conv_f32_any; 118x20x29x34 -> 225, 3x3 115, on k_conv2d_f32_dma 106)
            if (form.ti == 4 && form.tj == 2 && !quads(q[0].strips)) continue;
            const double time = estimate(form, q, n, cus) * (strips > 1 ? 1.02 : 1.0);
            if (time < form.time) {
               form.time = time;
               form.strips = strips;
            } else if (strips > form.strips + 1) {
               break;
            }
         }
         if (form.strips > 0 && (form.time < best.time || (form.time == best.time && best.ti > 0 && candidates[c].order < order))) {
            best = form;
            order = candidates[c].order;
         }
      }
      return best;
   }

   // Microseconds of a form on n images. A workgroup that is alone on its compute unit waits for memory in front of its loop,
   // once per slot and once per step, and for its stores behind it; workgroups that share one wait for each other's matrix
   // instructions (96 cycles a tile and step), operands, stores and conversions. A fit to 1760 timings of 201 convolutions over the ranges
   // of perf/cases.py (8.4 % rms; the form it picks is 1.1 % behind the best one in the mean).
   // q: of each kind of phases
   double estimate(const Form &f, const Panels *q, size_t n, int cus)
   {
      ++evaluated;
      int cells = 0;
      for (int k = 0; k < kinds; ++k) cells = q[k].cells > cells ? q[k].cells : cells;
      const int by_registers = resident_of(f.ti, f.tj, f.wo), by_lds = (int)MAX_LDS / (table_bytes(f.cs) + (slots(f.cs) > 1 ? 2 : 1) * slot_bytes(cells, f.cs));
      Sum s(*this, f, cus, by_lds < by_registers ? by_lds : by_registers, quads(q[0].strips));
      for (int k = 0; k < kinds; ++k) s.add(k, ((int)n * q[k].strips * q[k].PHW + f.pixels() - 1) / f.pixels(), q[k].cells);
      return s.time();
   }

   // The best form with slots of 8 channels, below other_us: strided layers, whose patches are too large for more (8x8 pixels under a 3x3
   // kernel of stride 2 read 17x17 cells, of 16 channels more than the 256 that the threads of a workgroup carry).
   Form choose_eights(size_t n, int cus, double other_us)
   {
      static const int forms[][3] = {{2, 2, 2}, {4, 4, 2}, {3, 4, 2}, {4, 2, 2}, {1, 2, 2}, {2, 4, 2}, {1, 4, 2}};
      Form best{0, 0, 0, 0, 0, other_us};
      if (pieces * 16 > ((size_t)1 << 29) || rows || nphases != 1 || chunks[0] < 4) return best;
      for (int t = 0; t < 3; ++t) least_cells[t][0] = cells_at_least(p.phase[0], 64 << t);
      for (const auto &f : forms) {
         if (f[0] > 1 && f[2] * (f[0] - 1) >= octiles) continue;      // tiles of nothing
         Form form{f[0], f[1], f[2], 8, 0, 0.0};
         if (least_cells[tile_of(form)][0] > cells_of(form) || least_time(form, n, cus) >= best.time) continue;
         form.time = HUGE_VAL;
         Strips &s = strips_seen[tile_of(form)];
         for (int strips = 1; strips <= MAX_STRIPS; ++strips) {
            if (strips > s.seen) look_at(s, form.pixels(), strips);
            const Panels &q = s.panels[strips - 1][0];
            if (s.cells[strips - 1] == 0 || q.cells > cells_of(form)) continue;
            if (table_bytes(8) + 2 * (long)slot_bytes(q.cells, 8) > MAX_LDS || (double)n * q.strips * q.PHW > (double)(1 << 30)) continue;
            if (form.ti == 4 && form.tj == 2 && !quads(q.strips)) continue;
            const double time = estimate(form, &q, n, cus) * (strips > 1 ? 1.02 : 1.0);
            if (time < form.time) {
               form.time = time;
               form.strips = strips;
            } else if (strips > form.strips + 1) {
               break;
            }
         }
         if (form.strips > 0 && form.time < best.time) best = form;
      }
      return best;
   }

   // All phases of a stride of 2 x 2 by one workgroup: the layer as a single phase whose patch is what the four read. False where
   // that is not possible.
   static bool together(const ConvProblem &p, ConvProblem &u)
   {
      if (p.nphases != 4 || p.sh != 1 || p.sw != 1) return false;
      u = p;
      u.nphases = 1;
      ConvPhase &f = u.phase[0];
      int below = 0, right = 0;
      for (int i = 0; i < 4; ++i) {
         const ConvPhase &q = p.phase[i];
         if (q.oys != 2 || q.oxs != 2 || q.oy0 != i / 2 || q.ox0 != i % 2) return false;
         if (q.OH > f.OH) f.OH = q.OH;
         if (q.OW > f.OW) f.OW = q.OW;
         if (q.ph > f.ph) f.ph = q.ph;
         if (q.pw > f.pw) f.pw = q.pw;
         if ((q.KH - 1) * p.dh - q.ph > below || i == 0) below = (q.KH - 1) * p.dh - q.ph;
         if ((q.KW - 1) * p.dw - q.pw > right || i == 0) right = (q.KW - 1) * p.dw - q.pw;
      }
      // (rows and columns of the patch as a kernel without dilation)
      f.KH = f.ph + below + 1;
      f.KW = f.pw + right + 1;
      u.dh = u.dw = 1;
      return f.KH >= 1 && f.KW >= 1;
   }

   // The best form with a phase per wavefront, below other_us; this: the plan of together()'s layer, apart: the one of the four phases.
   Form choose_together(const SplitPlan &apart, size_t n, int cus, double other_us)
   {
      static const int forms[][2] = {{4, 4}, {2, 4}, {3, 4}, {1, 4}};
      Form best{0, 0, 0, 0, 0, other_us};
      if (apart.pieces * 16 > ((size_t)1 << 29)) return best;
      bool even = true;
      int most = 0, all = 0;
      for (int i = 0; i < 4; ++i) {
         even = even && apart.chunks[i] == apart.chunks[0];
         most = apart.chunks[i] > most ? apart.chunks[i] : most;
         all += apart.steps[i];
      }
      one_for_all = true;
      chunks[0] = 4 * most;      // (of the tables of offsets, one for each phase)
      steps[0] = (all + 3) / 4;
      least_cells[0][0] = cells_at_least(p.phase[0], 64);
      Strips &s = strips_seen[0];      // (all these forms have tiles of 64)
      for (const auto &f : forms) {
         if (f[0] > 1 && f[0] - 1 >= octiles) continue;      // tiles of nothing
         for (int cs = 16; cs <= 32; cs *= 2) {
            // every wavefront comes to the same barriers: steps end with slots, or all alike
            bool fits = true;
            for (int i = 0; i < 4; ++i) fits = fits && (slots(cs) == 1 || (cs / 8 * apart.chunks[i] >= 4 && (even || cs / 8 * apart.chunks[i] % 4 == 0)));
            Form form{f[0], f[1], TOGETHER, cs, 0, 0.0};
            if (!fits || least_cells[0][0] > cells_of(form) || least_time(form, n, cus) >= best.time) continue;
            form.time = HUGE_VAL;
            for (int strips = 1; strips <= MAX_STRIPS; ++strips) {
               if (strips > s.seen) look_at(s, form.pixels(), strips);
               const Panels &q = s.panels[strips - 1][0];
               // (strips of a few columns: 192x224x13x13 -> 170, 2x2 s2 on strips of one 141 us, 106 apart)
               if (strips > 1 && q.ws < 8) break;
               if (s.cells[strips - 1] == 0 || q.cells > cells_of(form)) continue;
               if (table_bytes(cs) + (slots(cs) > 1 ? 2 : 1) * (long)slot_bytes(q.cells, cs) > MAX_LDS || (double)n * q.strips * q.PHW > (double)(1 << 30)) continue;
               const double time = estimate(form, &q, n, cus) * (strips > 1 ? 1.02 : 1.0);
               if (time >= form.time) continue;
               form.time = time;
               form.strips = strips;
            }
            if (form.strips > 0 && form.time < best.time) best = form;
         }
      }
      return best;
   }
   // Whether four pixels of two phases are stored at once: two neighbouring columns of each.
   bool pairs() const { return p.phase[0].OW % 4 == 0 && p.OW0 == 2 * p.phase[0].OW; }

private:
   const ConvProblem &p;

   struct Strips {
      int seen;                            // strips looked at: 1 .. seen
      int cells[MAX_STRIPS];               // most of any phase, 0: not possible
      Panels panels[MAX_STRIPS][MAX_PHASES];      // of each kind of phases
   };
   Strips strips_seen[3];                  // tiles of 64, 128 and 256 pixels
   int least_cells[3][MAX_PHASES];         // of each kind of phases
   static int tile_of(const Form &f) { return f.pixels() == 64 ? 0 : f.pixels() == 128 ? 1 : 2; }

   // Cells of the patch of bp pixels, whatever the strips: r rows of pixels of bp / r columns read ((r - 1) sh + h) x ((bp / r - 1) sw + w)
   // cells, h x w under one pixel; the smallest product over all real r (rounded down, and by 1 for the square roots).
   int cells_at_least(const ConvPhase &f, int bp) const
   {
      const double h = (double)(f.KH - 1) * p.dh + 1, w = rows ? 1.0 : (double)(f.KW - 1) * p.dw + 1, sh = p.sh < h ? p.sh : h, sw = rows ? 1.0 : p.sw < w ? p.sw : w;
      const double root = std::sqrt((h - sh) * (w - sw)) + std::sqrt(bp * sh * sw), cells = root * root;
      return cells < 1e6 ? (int)cells - 1 : 1000000;
   }

   void look_at(Strips &s, int bp, int strips)
   {
      int most = 0;
      for (int k = 0; k < kinds; ++k) {
         Panels &q = s.panels[strips - 1][k];
         if (!panels(q, kind[k], bp, strips)) {
            most = 0;
            break;
         }
         most = q.cells > most ? q.cells : most;
      }
      s.cells[strips - 1] = most;
      s.seen = strips;
   }

   struct Sum {
      const SplitPlan &l;
      const Form &f;
      int cus, resident, pieces, blocks, nslots;
      double store_alone, store, tiles = 0.0, alone = 0.0, work = 0.0;
      Sum(const SplitPlan &l, const Form &f, int cus, int resident, bool quads) : l(l), f(f), cus(cus), resident(resident)
      {
         pieces = f.ti * f.tj;
         blocks = (l.octiles + f.beside() * f.ti - 1) / (f.beside() * f.ti) * l.p.groups;
         nslots = l.slots(f.cs);
         store_alone = l.nphases > 1 || (l.one_for_all && !quads) ? 280.0 : quads ? 0.0 : 292.0;
         store = l.nphases > 1 ? 259.0 : quads ? 0.0 : l.one_for_all ? 259.0 : 176.0;
      }
      void add(int k, int pixel_tiles, int cells)
      {
         const int steps = l.steps[l.kind[k]];
         const double mma = 96.0 * steps * pieces, reads = (double)steps * (f.ti + f.tj), items = (double)cells * (f.cs / 8) / THREADS;
         const double t = (double)pixel_tiles * blocks * l.count[k];
         const double one = 3344.0 + (287.0 + store_alone) * pieces + nslots * (1053.0 + 785.0 * items) + 100.0 * reads + 0.579 * mma;
         if (one > alone) alone = one;
         work += t * (0.889 * mma + 33.5 * reads + (151.0 + store) * pieces + 598.0 * nslots * items + 527.0);
         tiles += t;
      }
      static double up(double v)
      {
         const double whole = (double)(long long)v;
         return whole < v ? whole + 1.0 : whole;
      }
      double time() const
      {
         const double per_cu = tiles / cus, rounds = per_cu / resident, whole = rounds + 0.895 * (up(rounds) - rounds);
         const double waits = alone * (whole > 1.0 ? whole : 1.0), busy = up(per_cu) * work / tiles;
         const double w2 = waits * waits, b2 = busy * busy;
         // (phases of unequal length, 3x3 s2: the same estimate was 1.25 to 1.5 times too short on 94 timings; with 1.4 the layers it takes of 190
         // random ones are 0.96 to 1.75 times k_conv_f32_any's time, with 1.35 0.94)
         const ConvPhase &q0 = l.p.phase[0], &q1 = l.p.phase[l.nphases - 1];
         // A phase per wavefront: 1.24 times what is estimated in the mean over 290 timings of 47 layers, even phases or not (14 % rms; what is
         // picked is 2.2 % behind the best of these forms in the mean): each wavefront takes in weights of its own.
         const double uneven = l.one_for_all ? 1.25 : q0.KH * q0.KW != q1.KH * q1.KW ? 1.4 : 1.0;
         const double us = std::sqrt(std::sqrt(w2 * w2 + b2 * b2)) / 2100.0 * uneven + 3.0;
         // (128 channels x 64 pixels ask for twice the weights per matrix instruction: over 221 layers of 15 to 700 us on which forms are close, each form timed, this
         // one takes 1.085 times what is estimated, 128 x 128 1.045 times, at every size. Of 84 other layers whose form changes by the 1.03, 25 of them above
         // 150 us, 0.975 times the time in the mean, 5 longer by more than 2 %, 1.043 at most. With 1.04 12x50x88x65 -> 194, 3x3 s2 35.4 -> 45.5.)
         return f.ti == 4 && f.tj == 2 ? 1.03 * us : us;
      }
   };

   // What the estimate cannot be below, whatever the strips: every pixel once, the fewest cells, the better kind of stores.
   double least_time(const Form &f, size_t n, int cus) const
   {
      Sum s(*this, f, cus, resident_of(f.ti, f.tj, f.wo), quads(1) || quads(2));
      for (int k = 0; k < kinds; ++k) s.add(k, (int)(((double)n * p.phase[kind[k]].OH * p.phase[kind[k]].OW + f.pixels() - 1) / f.pixels()), least_cells[tile_of(f)][k]);
      return s.time();
   }
};

}  // namespace sofie
