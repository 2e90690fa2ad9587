// Types shared by the translation units of the implicit-GEMM convolution (conv_igemm.hip: the float32
// kernels and the launch planning; conv_igemm_bf16.hip: the bf16-first kernels of the optional
// reduced-precision mode).
#pragma once
#include "tt_common.h"

namespace ttc {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;
constexpr int kBKQ = 4;          // k-quads per chunk (BK = 16)
constexpr int kInvalid = -(1 << 20);

// One entry per reduction index k (padded with never-valid entries to a whole chunk).
struct KEntry {
  int off;   // element offset added to the pixel's base offset (tap-mask tables: byte offset, biased to be >= 0)
  int dhw;   // (row step & 0xffff) | (column step << 16), both signed 16 bit (tap-mask tables: tap number; 31, or 63 with the 64-bit mask, = padding)
};

typedef int intx2 __attribute__((ext_vector_type(2)));
typedef const intx2 __attribute__((address_space(4))) * ConstKTab;   // constant address space: scalar (s_load) access

// What a launch does to a value between its accumulator and memory, beside the bias:
//   v = acc + bias;  v = (v - mean) * (gamma / sd) + beta  (norm);  v = v + res[same element];
//   v = maximum(v, 0), NaN kept  (relu);  v = v * (mask[same element] > 0)
// -- forward, the evaluation-mode BatchNorm, residual add and ReLU behind a convolution; backward, the
// gradient that has already arrived for x added to this one (res) and the backward of the ReLU that
// made x (mask) -- in the order and with the roundings of the kernels they stand in for.  `on` == 0:
// none of it.  Bound by memory: the three separate launches read and wrote y up to seven times over (a
// ResNet-50 evaluation pass at batch 64 in bf16 arithmetic spent half its time in them: 5.50 ms, 3.37 ms with
// this; 184 launches become 60, which at batch 2 takes 3.37 ms to 2.66).  Backward, the accumulation and
// the mask behind a residual block's input gradient were seven tensor passes and are three: with the residual
// add and the masks of batchnorm.hip, a ResNet-50 training step at batch 64 takes 20.53 ms for 21.97, at
// batch 32 in bf16 arithmetic 9.64 for 10.27.
struct Epilogue {
  const float *mean, *var, *gamma, *beta;   // [G*I] each; gamma / beta may be null
  const float* res;                         // laid out as `out`, or null
  const float* mask;                        // likewise
  float eps;
  int norm, relu, on;
};

struct Igemm {
  const float* src;
  const floatx4* wp;     // [G][KQ][Ipad] x 4 floats
  const KEntry* ktab;    // [KQ*4]
  const float* bias;     // [G*I] or null
  float* out;
  int I, Ipad, KQ, M;
  tt::FastDiv divUV, divV;   // m -> (n, u, v)
  int su, bh, sv, bw;        // ih0 = u*su + bh, iw0 = v*sv + bw
  int Hlim, Wlim, srcRow;
  int srcStrideN, srcStrideG;
  int outStrideN, outStrideG, outStrideI, outRow;
  int ou, ouh, ov, ovw;      // output row = u*ou + ouh, column = v*ov + ovw
  int tilesI;                // row tiles per group
  int tiles;                 // tilesI * pixel tiles
  // forward launches whose weight rows are a multiple of 4 long read the weights in place (a
  // row of w is already k-major): row stride in floats, 0 = use the repacked copy in wp
  const float* wraw;
  int wRowStride;
  // How the gathered operand is addressed:
  //   kModeCompare: 64-bit addresses, bounds compared per element (any geometry, any size)
  //   kModeGemm   : 1x1, stride 1, no padding: the operand is the [k][pixel] matrix of each image
  //                 itself; 16-byte buffer loads along pixels, kStride elements between k rows
  //   kModeTapMask: buffer loads; per tile every lane keeps one bit per tap (TB x TC <= 31 taps)
  //                 telling whether that tap falls outside the image for its pixel
  //   kModeTapMask64: the same with a 64-bit mask (32 .. 63 taps: 7x7 kernels), one 64-bit shift
  //                 per element instead of a 32-bit one
  // The two buffer modes address relative to the first image of the tile with 32-bit byte
  // offsets; the host selects them only when those stay below 2 GiB.
  int mode;
  int kStride, Kred;
  int TB, TC, stepH, stepW;  // tap window and steps of the table (tap-mask mode)
  int voffBias;              // elements added to every lane offset so that it is never negative
  long long srdBias;         // elements subtracted from the buffer base to make up for all biases
  const void* wbuf;          // buffer modes: base of the weight operand (wp or wraw)
  // buffer-mode input gradients of 1x1 layers read w[k][c] in place, transposed: row i of the
  // GEMM is column c of w, so lanes (rows) are contiguous and k strides by wTransStride = C/groups
  int wTransStride;
  // dense input-gradient launches only (all stride-parity classes as rows of one GEMM):
  // row i -> {element offset c*Hx*Wx + ch*Wx + cw, ch, cw, c}; output bounds outH x outW
  const int4* rowtab;
  int outH, outW;
  // strided 1x1 input gradients: only one pixel of every sh x 2 cell of dx has a tap.  > 0: the
  // launch stores each value together with the zero to its right (one 8-byte store) and zero
  // pairs into the cellFill - 1 rows below, so dx needs no clearing beforehand
  int cellFill;
  // stream-K launches only: the tiles*chunks reduction steps are dealt evenly to the blocks
  int skDpTiles;             // tiles [0, skDpTiles) are computed whole, block b takes b, b+blocks, ...
  int skBlocks;              // blocks that share the remaining tiles' reduction steps
  long long skIters;         // (tiles - skDpTiles) * (KQ / kBKQ)
  floatx4* skPartial;        // [skBlocks][acc float4s per thread][256] partial accumulators, one slot per block
  unsigned* skFlags;         // [block] = skEpoch once the block's partial is in memory
  unsigned skEpoch;          // differs from launch to launch, so the flags never need clearing
  unsigned* skError;         // one word in pinned host memory: set when a wait for a flag ran out
  Epilogue epi;
  // float32 launches of the three-term kernels: the weights as they came, element i*wI + c*wC + w0 + b*wRow + t*wCol
  // for row i, channel c and tap (b, t); null otherwise
  const float* w;
  int wI, wC, w0, wRow, wCol;
};


// Several data-parallel launches in one grid (the stride-parity classes of a strided input
// gradient): blocks [first[i], first[i+1]) belong to launch i.  One grid instead of a short
// launch per class, each with its own ramp-up and tail.
constexpr int kMaxMulti = 4;
struct IgemmMulti {
  Igemm c[kMaxMulti];
  int first[kMaxMulti + 1];
  int n;
};

// stream-K flags: one word per block.  A wait that runs out (about four seconds of polling: a block
// that was never scheduled, i.e. a grid that does not fit the device at two blocks per CU next to
// foreign work) is reported through a word in pinned host memory, which the host reads after its
// next stream synchronisation without any device operation.
constexpr int kSkFlagWords = 4096, kSkSpinLimit = 1 << 22;

constexpr int kModeCompare = 0, kModeGemm = 1, kModeTapMask = 2, kModeTapMask64 = 3;
constexpr int kSrdFlags = 0x00020000;        // raw buffer, 32-bit data format
constexpr int kSrdRecords = 0x7fffffff;      // offsets with bit 31 set are out of range and read 0

__device__ __forceinline__ float as_float(unsigned v) { return __builtin_bit_cast(float, v); }

// Per-row constants of the epilogue for the BM rows of a tile, {mean, gamma / sd, beta, bias} each an
// array of BM in LDS: one thread computes a row's once (a square root and a division) while the tile's
// first loads are in flight, instead of every lane for each of its rows at the end.  The caller's next
// barrier publishes them.  Without a bias or a normalisation the constants leave a value as it is:
// v + -0, (v - 0) * 1 + -0.
template <int BM>
__device__ __forceinline__ void epilogue_constants(const Igemm& p, int first_channel, int i0, int tid, float* lds) {
  const Epilogue& e = p.epi;
  if (tid < BM) {
    const int c = first_channel + min(i0 + tid, p.I - 1);
    float m = 0.f, k1 = 1.f, k0 = -0.f;
    if (e.norm) {
      const float sd = __fsqrt_rn(__fadd_rn(e.var[c], e.eps));
      m = e.mean[c];
      k1 = __fdiv_rn(e.gamma ? e.gamma[c] : 1.0f, sd);
      k0 = e.beta ? e.beta[c] : 0.0f;
    }
    lds[tid] = m;
    lds[BM + tid] = k1;
    lds[2 * BM + tid] = k0;
    lds[3 * BM + tid] = p.bias ? p.bias[c] : -0.f;
  }
}

// Stores one wave's MT x NT accumulators through the epilogue.  `row0` is the wave's first row inside
// the tile; accumulator register r of a 32x32 tile holds row 8*(r/4) + 4*h + r%4.  A 32-row strip's
// residual and mask values are all fetched before its first store (loads and stores share one in-order
// counter).  Rows and pixels past the end re-read the last row / pixel 0 and are never stored.
template <int BM, int MT, int NT>
__device__ __forceinline__ void store_through_epilogue(const Igemm& p, const floatx16 (&acc)[MT][NT], const uint32_t (&obase)[NT],
                                                       const bool (&mok)[NT], int i0, int row0, int h, const float* lds) {
  const float floor_ = p.epi.relu ? 0.f : -__builtin_huge_valf();
#pragma unroll
  for (int x = 0; x < MT; ++x) {
    const int r0 = row0 + 32 * x + 4 * h;   // + 8*q + j inside the tile
    float rs[NT][16], ms[NT][16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        rs[y][r] = -0.f;   // v + -0 is v
        ms[y][r] = 1.f;
      }
    }
    auto fetch = [&](const float* __restrict__ from, float (&to)[NT][16]) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t ioff = (uint32_t)(min(i0 + r0 + 8 * (r >> 2) + (r & 3), p.I - 1) * p.outStrideI);
#pragma unroll
        for (int y = 0; y < NT; ++y) to[y][r] = from[obase[y] + ioff];
      }
    };
    if (p.epi.res) fetch(p.epi.res, rs);
    if (p.epi.mask) fetch(p.epi.mask, ms);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 m4 = *reinterpret_cast<const floatx4*>(lds + r0 + 8 * q);
      const floatx4 s4 = *reinterpret_cast<const floatx4*>(lds + BM + r0 + 8 * q);
      const floatx4 b4 = *reinterpret_cast<const floatx4*>(lds + 2 * BM + r0 + 8 * q);
      const floatx4 z4 = *reinterpret_cast<const floatx4*>(lds + 3 * BM + r0 + 8 * q);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + r0 + 8 * q + j;
        if (i < p.I) {
          const uint32_t ioff = (uint32_t)(i * p.outStrideI);
#pragma unroll
          for (int y = 0; y < NT; ++y) {
            float v = acc[x][y][4 * q + j] + z4[j];
            v = fmaf(v - m4[j], s4[j], b4[j]) + rs[y][4 * q + j];
            v = (v > floor_ || v != v) ? v : floor_;
            v *= ms[y][4 * q + j] > 0.f ? 1.f : 0.f;
            if (mok[y]) p.out[obase[y] + ioff] = v;
          }
        }
      }
    }
  }
}

// Float32 launches on three bfloat16 terms multiply both operands by kLift on their way in and the sums by kLower
// on their way out: exact, and what a term holds then reaches down to the least float32, 2^-149 (a bfloat16 has no bit
// below 2^-133, so that without it operands under 2^-110 lost bits and those under 2^-134 all of them: 64 products
// of 2^-126 and 2^60 were off by 7e-4, of 2^-135 and 2^60 they were zero).  One vector instruction per value:
// 512 to 256 channels 1x1, 28x28 at batch 64, 95 us without, 98 with; 128 channels 3x3, 16x16 at batch 128, 69 and 69.
// What it takes from the other end -- operands from 2^104, sums from 2^80 on -- comes out as an infinity or NaN, like
// everything that is not finite itself, and such sums are formed again (float32_sums).
constexpr float kLift = 0x1p24f, kLower = 0x1p-48f;

// Whether a lane's sums hold an infinity or NaN.  Two values an instruction (v_maximum3_f32, which keeps NaN).
template <int MT, int NT>
__device__ __forceinline__ bool not_finite(const floatx16 (&acc)[MT][NT]) {
  float most = 0.f;
#pragma unroll
  for (int x = 0; x < MT; ++x)
#pragma unroll
    for (int y = 0; y < NT; ++y)
#pragma unroll
      for (int r = 0; r < 16; r += 2)
        most = __builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_fabsf(acc[x][y][r]), __builtin_fabsf(acc[x][y][r + 1])), most);
  return !(most <= 3.402823466e38f);
}

// The operands of a wave's tiles as they lie in memory: lane l32 + 32*h holds row l32 of every row tile and pixel l32
// of every pixel tile.  Tap (r, s) of channel c is w[x][c*wC + r*wRow + s*wCol] and pixel row ih[y] + r*dh, column
// iw[y] + s*dw of the plane src[y] + c*plane, zero outside it.
template <int MT, int NT>
struct WaveOperands {
  const float* w[MT];
  const float* src[NT];
  int ih[NT], iw[NT];
  int R, S, wC, wRow, wCol, dh, dw, H, W, srcRow;
  long long plane;
};

// Their sums over the channels [c0, c1) on the float32 matrix instructions, what launches without terms compute: for
// the few waves of a launch in three terms that not_finite stops.  Operands come straight from memory, four
// steps' loads in flight: launches whose every sum is infinite or NaN take 368 us for 128 on the float32 instructions alone
// (512 to 256 channels 1x1, 28x28 at batch 64) and 224 for 93 (128 channels 3x3, 16x16 at batch 128); summed
// one by one, in float64, they took 26.8 and 13.3 ms.  One infinite pixel in every image costs 230 and 214 us, then 9.9
// and 7.4 ms.
template <int MT, int NT>
__device__ __forceinline__ void float32_sums(floatx16 (&acc)[MT][NT], const WaveOperands<MT, NT>& o, const int c0, const int c1, const int h) {
#pragma unroll
  for (int x = 0; x < MT; ++x)
#pragma unroll
    for (int y = 0; y < NT; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][y][r] = 0.f;
  constexpr int kSteps = 4;
  for (int r = 0; r < o.R; ++r)
    for (int s = 0; s < o.S; ++s) {
      const float* w[MT];
      const float* src[NT];
      bool inside[NT];
#pragma unroll
      for (int x = 0; x < MT; ++x) w[x] = o.w[x] + r * o.wRow + s * o.wCol;
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        const int ih = o.ih[y] + r * o.dh, iw = o.iw[y] + s * o.dw;
        inside[y] = (unsigned)ih < (unsigned)o.H && (unsigned)iw < (unsigned)o.W;
        src[y] = o.src[y] + (inside[y] ? (long long)ih * o.srcRow + iw : 0);
      }
      for (int c = c0; c < c1; c += 2 * kSteps) {   // lanes 0-31 hold a step's first channel, lanes 32-63 its second
        float a[kSteps][MT], b[kSteps][NT];
#pragma unroll
        for (int k = 0; k < kSteps; ++k) {
          const int ch = c + 2 * k + h;
          const long long at = min(ch, c1 - 1);
#pragma unroll
          for (int x = 0; x < MT; ++x) a[k][x] = w[x][at * o.wC];
#pragma unroll
          for (int y = 0; y < NT; ++y) b[k][y] = src[y][at * o.plane];
#pragma unroll
          for (int x = 0; x < MT; ++x) a[k][x] = ch < c1 ? a[k][x] : 0.f;
#pragma unroll
          for (int y = 0; y < NT; ++y) b[k][y] = ch < c1 && inside[y] ? b[k][y] : 0.f;
        }
        // eight products add up on their own first: shorter chains, and smaller errors, than one over the whole reduction
#pragma unroll
        for (int x = 0; x < MT; ++x)
#pragma unroll
          for (int y = 0; y < NT; ++y) {
            floatx16 part = {};
#pragma unroll
            for (int k = 0; k < kSteps; ++k) part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k][x], b[k][y], part, 0, 0, 0);
            acc[x][y] += part;
          }
      }
    }
}

// The bf16-first kernels (conv_igemm_bf16.hip).  `supported` tells whether they take launch `p`
// (tile rows `bm` as planned by the caller); `launch` enqueues it on the library stream.
bool bf16_first_supported(const Igemm& p, int groups, int bm);
void bf16_first_launch(const Igemm& p, int groups, int bm, hipStream_t st);


// The channel-last kernels (conv_hwc.hip): one group, operands rounded to bfloat16.  x is [N][C][H][W], the
// result [N][I][P][Q]; output pixel (u, v) reads input rows u*sh - ph + r*dh (ph, pw may be negative).
// dgrad: w is [C][I][R][S] with its taps reversed instead of [I][C][R][S].
struct HwcConv {
  int N, C, H, W, I, P, Q, R, S, sh, sw, ph, pw, dh, dw;
  bool dgrad;
};
// Whether they take it; `always`: also where the size rule prefers the other kernels (small test shapes).
bool hwc_supported(const HwcConv& c, bool always);
size_t hwc_workspace(const HwcConv& c);
// Enqueues the call; `plan8` as tt_conv2d_last_launch reports it.
int hwc_conv(const HwcConv& c, const float* x, const float* w, const float* bias, float* out, const Epilogue* epi, int prof_id,
             int* plan8);
// Enqueues the sum of `splits` partial results in order, each laid out as p.out (one group), and the launch's
// bias and epilogue.
int add_partials(const Igemm& p, const float* partial, int splits);

// The kernel body of conv_igemm_kernel.h in one arithmetic (conv_igemm_launch.h).  launch: `bm` x `bn` is
// the tile the caller planned; `sk_blocks` > 0 asks for the persistent (stream-K) grid, which is launched
// only if the device holds that many blocks at once (`forced_occupancy` >= 0 replaces what the device
// says: tests); returns whether it was.  min_resident_blocks: resident blocks per compute unit of its
// stream-K kernels, the smallest over every instantiation.
struct IgemmUnit {
  bool (*launch)(const Igemm& p, int groups, int sk_blocks, int bm, int bn, int forced_occupancy, hipStream_t st);
  void (*launch_multi)(const IgemmMulti& m, int groups, int bm, int bn, hipStream_t st);
  int (*min_resident_blocks)();
};
const IgemmUnit& igemm_f32_unit();
const IgemmUnit& igemm_bf16_unit();
const IgemmUnit& igemm_bf16x3_unit();
const IgemmUnit& igemm_epi_f32_unit();   // for launches with Igemm::epi.on
const IgemmUnit& igemm_epi_bf16_unit();
const IgemmUnit& igemm_epi_bf16x3_unit();

}  // namespace ttc
