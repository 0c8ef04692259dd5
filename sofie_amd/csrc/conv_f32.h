// fp32 convolutions: what their kernels share.
#pragma once
#include "common.h"

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

// Runs the problem on k_conv_f32_any (conv_f32_any.hip) or k_conv_f32_split; *done stays false where they do not take it, or where
// the former's estimate is above the microseconds of the caller's other way. split_only: not on the former.
int conv_f32_any(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done, bool split_only = false);

// Runs the problem on k_conv_f32_split (conv_f32_split.hip); *done stays false where it does not take it, or where its estimate is above
// the microseconds of the caller's other way.
int conv_f32_split(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done);

// The same for k_conv_f32_short (conv_f32_short.hip).
int conv_f32_short(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done);

}  // namespace sofie
