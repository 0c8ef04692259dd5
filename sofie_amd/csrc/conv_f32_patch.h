// k_conv_f32_split (conv_f32_split.hip): how many rows of input a tile reads. The arithmetic alone, also for a host program that
// checks it against every tile.
#pragma once

namespace sofie {

// Most input rows under bp consecutive pixels. Pixels run over panels (strips of images) of OH x ws, row by row; with `apart` a panel is
// filled up to whole tiles. A panel's input has (OH - 1) * sh + (KH - 1) * dh + 1 rows, panels lie one below the other.
inline long split_patch_rows(int bp, int ws, long panel_pixels, int OH, int sh, int KH, int dh, bool apart)
{
   // rows of output a tile touches at most (whole ones where they divide a tile: panels are whole rows), panels it reaches into at most,
   // and what lies between two rows of it
   const long rows = bp % ws == 0 ? bp / ws : (bp + ws - 2) / ws + 1, cross = apart ? 0 : (bp + panel_pixels - 2) / panel_pixels;
   const long halo = (long)(KH - 1) * dh + 1, between = halo > sh ? halo : sh, more = rows - 1 > cross ? rows - 1 - cross : 0;
   return more * sh + cross * between + halo;
}

}  // namespace sofie
