"""The rows of input a tile of k_conv_f32_split keeps in LDS (sofie_amd/csrc/conv_f32_patch.h), worked out on the host by the header the
kernel's launcher uses, against the rows that every tile of a layer reads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "conv_f32_patch.h"
int main()
{
   long checked = 0, spare = 0;
   for (int bp : {64, 128, 256})
      for (int OH : {1, 2, 3, 7, 10, 28, 57})
         for (int ws : {1, 2, 5, 8, 17, 28, 56})
            for (int KH : {1, 2, 3, 5, 7})
               for (int dh : {1, 2, 3})
                  for (int sh : {1, 2, 3, 8})
                     for (int apart = 0; apart < 2; ++apart) {
                        const long full = (long)OH * ws, panel = apart ? (full + bp - 1) / bp * bp : full;
                        const long HP = (long)(OH - 1) * sh + (KH - 1) * dh + 1, rows = sofie::split_patch_rows(bp, ws, panel, OH, sh, KH, dh, apart);
                        const long P = panel * (4 + 2 * bp / panel);
                        long most = 0;
                        for (long p0 = 0; p0 < P; p0 += bp) {
                           long last = 0;
                           const long origin = p0 / panel * HP + p0 % panel / ws * sh;
                           for (long p = p0; p < p0 + bp && p < P; ++p)
                              if (p % panel < full) last = p / panel * HP + p % panel / ws * sh + (KH - 1) * dh + 1 - origin;
                           most = last > most ? last : most;
                        }
                        if (most > rows) return printf("%d %d %d %d %d %d %d: %ld > %ld\n", bp, OH, ws, KH, dh, sh, apart, most, rows), 1;
                        ++checked;
                     }
   printf("%ld\n", checked);
}
"""


def test_every_tile_reads_within_its_rows(tmp_path):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert int(out.stdout) == 3 * 7 * 7 * 5 * 3 * 4 * 2
