// fp32 convolutions: what their kernels share.
#pragma once
#include "common.h"
#include "conv_f32_problem.h"

namespace sofie {

// Runs the problem on k_conv_f32_any (conv_f32_any.hip), k_conv_f32_split or k_conv_f32_short; *done stays false where they do not take it,
// or where their estimates are above the microseconds of the caller's other way (HUGE_VAL: it has no estimate of that). SPLIT_ONLY: on
// k_conv_f32_split, if that is shorter than k_conv_f32_any by their estimates; SPLIT_DECLINED: the same call has come with SPLIT_ONLY before.
enum ConvWays { ALL_WAYS, SPLIT_ONLY, SPLIT_DECLINED };
int conv_f32_any(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done, ConvWays ways = ALL_WAYS);

// Runs the problem on k_conv_f32_split (conv_f32_split.hip); *done stays false where it does not take it, or where its estimate is above
// the microseconds of the caller's other way.
int conv_f32_split(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done);

// The same for k_conv_f32_short (conv_f32_short.hip).
int conv_f32_short(sofie_hip_ctx *ctx, const ConvProblem &p, double other_us, bool *done);

}  // namespace sofie
