// The kernels for convolutions of unit stride on three bfloat16 terms (conv_patch.hip).
#pragma once
#include "conv_igemm_common.h"

namespace ttc {

// x is [N][C][H][W], the result [N][I][P][Q]; output pixel (u, v) reads input rows u - ph + r*dh (ph, pw may be
// negative).  dgrad: w is [C][I][R][S] with its taps reversed instead of [I][C][R][S].
struct PatchConv {
  int N, C, H, W, I, P, Q, R, S, ph, pw, dh, dw;
  bool dgrad;
};
// f32: the call is one of float32 arithmetic (TT_CONV_MATH_F32), not of bf16x3: operands of any magnitude, infinities
// and NaN give what they give there.
bool patch_conv_takes(const PatchConv& c, bool f32);
size_t patch_workspace(const PatchConv& c);
// Enqueues the call; `plan8` as tt_conv2d_last_launch reports it.
int patch_conv_launch(const PatchConv& c, const float* x, const float* w, const float* bias, float* out, const Epilogue* epi,
                      bool f32, int prof_id, int* plan8);

}  // namespace ttc
