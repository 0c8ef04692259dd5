// What an fp32 convolution kernel is asked for: the arithmetic of a layer, without anything of the device.
#pragma once
#include <stddef.h>

namespace sofie {

// One plain correlation of an NCHW input: pixel (q, r) of OH x OW reads input rows q * sh - ph + a * dh, columns
// r * sw - pw + b * dw for the taps (a, b) of KH x KW, and is stored at row oy0 + q * oys, column ox0 + r * oxs of a plane
// of OH0 x OW0. Tap (a, b) is element (th0 + a * ths, tw0 + b * tws) of the KH0 x KW0 kernel in memory. A convolution is
// one of these, a transposed convolution one per output phase (oy mod stride, ox mod stride).
struct ConvPhase {
   int OH, OW, KH, KW, ph, pw;
   int th0, ths, tw0, tws;
   int oy0, oys, ox0, oxs;
};

struct ConvProblem {
   const float *x, *w, *bias;
   float *y;
   int N, C, H, W, OC, groups, sh, sw, dh, dw, relu;
   int KH0, KW0, OH0, OW0;
   int transposed;             // w is [C][OC/groups][KH0][KW0], else [OC][C/groups][KH0][KW0]
   int nphases;
   ConvPhase phase[4];
};

}  // namespace sofie
