// The kernels for convolutions on three bfloat16 terms that keep a patch of the source in LDS (conv_patch.hip).
#pragma once
#include "conv_igemm_common.h"

namespace ttc {

// A forward pass is one class of pixels, an input gradient one for each parity of its stride.  Pixel (n, u, v) of
// U x V reads source rows u - ph + r*dh, columns v - pw + s*dw for its R x S taps (ph, pw may be negative), tap (r, s)
// being element w0 + r*wRow + s*wCol of the kernel, and lands in row u*ou + ouh, column v*ov + ovw of its plane.
constexpr int kPatchClasses = 4;
struct PatchConvClass {
  int U, V, R, S, ph, pw, dh, dw, ouh, ovw, w0, wRow, wCol;
};
// The source is [N][C][H][W], the result [N][I][outPlane], its rows outRow long.  dgrad: w is [C][I][taps] instead of
// [I][C][taps].
struct PatchConv {
  int N, C, H, W, I, outPlane, outRow, ou, ov, taps;
  bool dgrad;
  int n;
  PatchConvClass c[kPatchClasses];
};
// f32: the call is one of float32 arithmetic (TT_CONV_MATH_F32), not of bf16x3: operands of any magnitude, infinities
// and NaN give what they give there.
bool patch_conv_takes(const PatchConv& c, bool f32);
size_t patch_workspace(const PatchConv& c);
// Enqueues the call; `plan8` as tt_conv2d_last_launch reports it.
int patch_conv_launch(const PatchConv& c, const float* x, const float* w, const float* bias, float* out, const Epilogue* epi,
                      bool f32, int prof_id, int* plan8);

}  // namespace ttc
