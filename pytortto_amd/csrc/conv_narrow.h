// The kernels for convolutions with few rows (conv_narrow.hip).
#pragma once
#include "conv_igemm_common.h"

namespace ttc {

// One stride-parity class of an input gradient (a forward pass is one class): pixel (n, u, v) of U x V reads
// source row u*su + bh + b*stepH, column v*sv + bw + c*stepW for its TB x TC taps, tap (b, c) being element
// (r0 + b*rs, s0 + c*ss) of the kernel, and lands in row u*ou + ouh, column v*ov + ovw.
struct NarrowClass {
  int U, V, M;
  tt::FastDiv divUV, divV, divTC, divTaps;   // (divTaps: set by the launch)
  int bh, bw, TB, TC, r0, s0, ouh, ovw;
  int block0;   // its first block (set by the launch)
};
constexpr int kNarrowClasses = 16;
struct NarrowConv {
  const float *src, *w, *bias;   // bias may be null
  float* out;
  int I, A, groups;              // rows and source planes of a group
  tt::FastDiv divA, divUnit;     // channels; steps of a unit of four taps (set by the launch)
  int wI, wA, wG, rs, ss, S;     // strides of w: row, plane, group; tap steps; kernel width
  int su, sv, stepH, stepW;
  int Hlim, Wlim, srcN, srcG, plane;
  int outN, outG, outI, outRow, ou, ov;
  bool gradient;                 // of the input
  int n;
  NarrowClass c[kNarrowClasses];
  Epilogue epi;
};
bool narrow_conv_takes(const NarrowConv& p, bool bf16);
int narrow_conv_launch(NarrowConv& p, bool bf16, int prof_id, int* plan8);   // plan8 as tt_conv2d_last_launch reports it

struct NarrowWgrad {
  const float *x, *dy;
  float *out, *part;
  int Kg, J, M, groups;
  tt::FastDiv divPQ, divQ, divRS, divS;
  int H, W, HW, PQ, R, S, sh, sw, ph, pw, dh, dw;
  int xN, xG, dyN, dyG, xBias;   // xBias = ph*W + pw
  int KT, JT, tilesI, tilesJ, splits, perSplit;   // set by narrow_wgrad_takes
};
bool narrow_wgrad_takes(NarrowWgrad& p, bool bf16);
size_t narrow_wgrad_workspace(const NarrowWgrad& p);
int narrow_wgrad_launch(NarrowWgrad& p, bool bf16);

}  // namespace ttc
