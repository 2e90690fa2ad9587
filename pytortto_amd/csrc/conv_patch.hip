// Convolutions whose operands travel as three bfloat16 terms and whose pixels reach consecutive ones of the source:
// forward passes of unit stride, input gradients of any (a strided one is a class of pixels for each parity of its
// stride, and each class is such a convolution; up to four).
//
//   D[i, m] = sum over channels c and taps t of  W[i][c][t] * X[pixel(m, t)][c]      (+ epilogue)
//
// The kernels that gather in place (conv_igemm_kernel.h) fetch a source element, write it to LDS and split
// it into its terms once per tap, and do so between barriers 24 matrix instructions apart: nothing overlaps
// with anything, and the matrix pipe is busy for a third of the time.  Here a block fetches the patch of the
// source that its pixels reach -- all taps of it -- once per sixteen channels, splits it once, and runs the
// taps out of LDS: a tap is a constant added to the address of a lane's pixel.  Between two barriers lie 24
// matrix instructions per wave for every tap (216 for a 3x3 kernel), and a source element is fetched 1.3 to
// 1.7 times instead of nine.  The weights are split and laid out once per call, in the order in which a
// wave's lanes hold them, and go from memory to registers without passing LDS.
//
// Measured, 3x3, forward: 160 to 192 channels 45x37 at batch 24 117 us (189 TFLOP/s of the product: its six matrix
// instructions run at 1.13 PFLOP/s, what a large bf16 product reaches here), 184 in the kernels that gather; 64
// channels 32x32 at batch 128 63 us (50 of them the product), 72; 128 channels 16x16 67, 98.  471 blocks,
// two on a compute unit, keep the matrix pipes busy for 52 % of the cycles at a clock that the device's power holds at
// 2.2 GHz; 256, or 512 that share their reductions, for 36 and 39 % at 2.4: there what a wave does between two chunks
// bounds it, and the sums' way through memory.
//
// Float32 arithmetic uses them too, where a call is large: the terms add up to the operands exactly, what is left out
// of a product is below half an ulp of it, and the error against float64 sums is 0.33 to 0.66 times that of the
// float32 instructions, which round twice as often (42 launches).  A ResNet-50 training step at batch 64 takes
// 19.43 ms for 20.27, a PreAct-ResNet-18 one at batch 128 4.81 for 5.35.  What three terms do not hold is summed
// again on the float32 instructions (not_finite).
//
// The pixels of a tile are consecutive pixels of the batch, whatever the image's shape.  Their source lies in
// a virtual image that holds the images of the batch below each other, each framed by what the taps reach
// outside it: virtual pixel (n*VR + j)*PW + k is row j + bh, column k + bw of image n, zero outside.  A
// pixel's taps are at fixed distances there, so the patch is one range of it.  Where two images' frames (or
// two rows') meet, they are zeros from either side, and share them.
#include <algorithm>
#include <initializer_list>
#include <utility>

#include "conv_igemm_common.h"
#include "conv_patch.h"

namespace {

using namespace ttc;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 16;              // channels of a chunk: the depth of one matrix step
constexpr int kTerms = 3;
constexpr int kUnit = 16 * kTerms;   // bytes of a patch pixel's eight channels.  48 bytes from lane to lane
                                     // spread eight lanes' 16-byte accesses over all banks, while the pixels are
                                     // consecutive: in a ResNet-50 step, of images 7 to 56 wide, 27 to 48 % of the LDS's
                                     // cycles are bank conflicts.  It is busy for 15 to 22 % of the kernel's, and bounds nothing
constexpr int kMaxTaps = 31;
// Taps of weights that a wave of the product reads past its own: two ahead of the one it multiplies, and an odd
// number of taps is rounded up to a pair, whose second tap fetches one more.
constexpr int kReadPast = 3;

// Eight float32 values as three vectors of bfloat16 terms that add up to them exactly: term i of a value is
// the bf16 nearest to what the terms before it leave.
__device__ __forceinline__ void split8(const float (&v)[8], uintx4 (&out)[kTerms]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float e = v[2 * q], o = v[2 * q + 1];
#pragma unroll
    for (int i = 0; i < kTerms; ++i) {
      const bf16x2 pair = {(__bf16)e, (__bf16)o};
      unsigned t = __builtin_bit_cast(unsigned, pair);
      asm("" : "+v"(t));   // or the compiler rounds the even value a second time, by itself
      out[i][q] = t;
      if (i < kTerms - 1) {
        e -= as_float(t << 16);
        o -= as_float(t & 0xffff0000u);
      }
    }
  }
}

// Which taps of the kernel the classes of a call run, for the layout of their weights: tap (r, s) of class k is
// element w0 + r*wRow + s*wCol of the kernel, its weights begin at wt (units of 16 bytes).
struct PatchTaps {
  int n;
  int taps[kPatchClasses], S[kPatchClasses], w0[kPatchClasses], wRow[kPatchClasses], wCol[kPatchClasses];
  size_t wt[kPatchClasses];
};

// ---- weights -> wt[32 rows][chunk][tap][term][lane], 16 bytes each: lane 32*h + l holds row l, channels 8h.. --
// forward: row k, w[k][c][tap];  input gradient: row c, channel k.  A block lays out one strip of 32 rows and
// sixteen channels for every class: reads runs of w, turns them in LDS, writes runs of wt.
template <bool DGRAD>
__global__ __launch_bounds__(kThreads) void patch_weights(const float* __restrict__ w, uintx4* __restrict__ wt, int rows, int chans,
                                                         int taps, tt::FastDiv divRun, int chunks, float lift, const PatchTaps classes) {
  extern __shared__ float strip[];   // [outer][run + 1]: forward 32 rows x 16 channels' taps, gradient 16 x 32 rows' taps
  const int chunk = blockIdx.x, r0 = blockIdx.y * 32, c0 = chunk * kBK;
  const int run = divRun.d;          // (DGRAD ? 32 : 16) * taps
  const int outer = DGRAD ? kBK : 32;
  for (int u0 = threadIdx.x; u0 < outer * run; u0 += 8 * kThreads) {   // eight loads in flight: small layers have few blocks
    float v[8];
    int at[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int u = u0 + e * kThreads;
      const int a = (int)tt::fd_div((uint32_t)u, divRun), b = u - a * run;
      const bool ok = a < outer && (DGRAD ? c0 + a < chans && r0 * taps + b < rows * taps : r0 + a < rows && c0 * taps + b < chans * taps);
      const size_t from = DGRAD ? ((size_t)(c0 + a) * rows + r0) * taps + b : ((size_t)(r0 + a) * chans + c0) * taps + b;
      at[e] = a < outer ? a * (run + 1) + b : -1;
      v[e] = ok ? w[from] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (at[e] >= 0) strip[at[e]] = v[e] * lift;
  }
  __syncthreads();
  for (int k = 0; k < classes.n; ++k) {
    const int mine = classes.taps[k], S = classes.S[k];
    uintx4* __restrict__ dst = wt + classes.wt[k] + ((size_t)blockIdx.y * chunks + chunk) * mine * (kTerms * 64);
    for (int u = threadIdx.x; u < mine * 64; u += kThreads) {
      const int tap = u >> 6, lane = u & 63, row = lane & 31, c = 8 * (lane >> 5);
      const int from = classes.w0[k] + tap / S * classes.wRow[k] + tap % S * classes.wCol[k];
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = DGRAD ? strip[(c + e) * (run + 1) + row * taps + from] : strip[row * (run + 1) + (c + e) * taps + from];
      uintx4 t[kTerms];
      split8(v, t);
#pragma unroll
      for (int i = 0; i < kTerms; ++i) dst[(tap * kTerms + i) * 64 + lane] = t[i];
    }
  }
}

// ---- the product -------------------------------------------------------------------------------------
struct PatchClass {
  int M;                     // pixels (n, u, v)
  tt::FastDiv divUV, divV;
  int bh, bw, ouh, ovw;      // tap 0 reads row u + bh, column v + bw; the result is row u*ou + ouh, column v*ov + ovw
  int taps, S;
  int PW, VR;                // the virtual image's pitch and rows per image
  tt::FastDiv divPW, divVR;
  int px;                    // pixels of the patch held in LDS
  int tapRow, tapCol;        // steps of a tap row / column in the patch, in bytes
  int dh, dw;                // the same in pixels of the source
  int w0, wRow, wCol;        // tap (r, s) is element w0 + r*wRow + s*wCol of the kernel
  int block0;                // its first tile
  size_t wt;                 // where its weights begin, units of 16 bytes
};
struct Patch {
  const float* src;
  const uintx4* wt;
  float* partial;      // splits > 1: [splits][elements of out] sums over a part of the chunks each
  long long outElems;
  int C, chunks, perSplit;
  int plane, image;    // bytes of a source plane, an image
  int maxPx;           // of the classes' patches
  int images;
  // float32 launches: the weights as they came, strides of a row and a channel; null otherwise
  const float* w;
  int wI, wC;
  int classes;
  PatchClass c[kPatchClasses];
};

// Tile 32*WM rows x 32*NT*(4/WM) pixels; every wave has 32 rows and NT x 32 pixels.  The patch has at most 128*IT
// pixels: a thread fetches and splits eight channels of IT of them.
template <int WM, int NT, int IT, bool EPI>
__global__ __launch_bounds__(kThreads, 2) void patch_product(const Igemm p, const Patch q) {
  constexpr int WN = 4 / WM, BM = 32 * WM, BN = 32 * NT * WN;
  extern __shared__ __align__(16) char lds[];   // [half][px] units; then the epilogue's constants
  float* const epi_lds = reinterpret_cast<float*>(lds + 2 * q.maxPx * kUnit);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int all = tt::xcd_remap((int)blockIdx.x, (int)gridDim.x);
  int ci = 0;
  while (ci + 1 < q.classes && all >= q.c[ci + 1].block0) ++ci;
  const PatchClass& k = q.c[ci];
  const int tile = all - k.block0, tilesI = p.Ipad / BM;
  const int i0 = (tile % tilesI) * BM;
  const int m0 = (tile / tilesI) * BN;
  const int q0 = (int)blockIdx.z * q.perSplit, q1 = min(q.chunks, q0 + q.perSplit);

  // pixel m is (n, u, v)
  auto split_pixel = [&](const uint32_t m, uint32_t& n, uint32_t& u, uint32_t& v) __attribute__((always_inline)) {
    n = tt::fd_div(m, k.divUV);
    v = m - n * k.divUV.d;
    u = tt::fd_div(v, k.divV);
    v -= u * k.divV.d;
  };
  auto virtual_pixel = [&](const uint32_t m, uint32_t& n) __attribute__((always_inline)) {
    uint32_t u, v;
    split_pixel(m, n, u, v);
    return (n * (uint32_t)k.VR + u) * (uint32_t)k.PW + v;
  };
  uint32_t n0;
  const uint32_t first = virtual_pixel((uint32_t)__builtin_amdgcn_readfirstlane(m0), n0);
  const __amdgpu_buffer_rsrc_t srd =
      __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)q.src + (long long)n0 * q.image), 0, kSrdRecords, kSrdFlags);

  // what this thread fetches: half `wave / 2` of the patch pixels it*128 + tid % 128
  const int half = wave >> 1, pp0 = tid & 127;
  const int at = (half * k.px + pp0) * kUnit;
  int voff[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int pp = it * 128 + pp0;
    const uint32_t v = first + (uint32_t)pp;
    const uint32_t row = tt::fd_div(v, k.divPW), n = tt::fd_div(row, k.divVR);
    const int ih = (int)(row - n * (uint32_t)k.VR) + k.bh, iw = (int)(v - row * (uint32_t)k.PW) + k.bw;
    const bool inside = pp < k.px && (unsigned)ih < (unsigned)p.Hlim && (unsigned)iw < (unsigned)p.Wlim && n < (uint32_t)q.images;
    voff[it] = inside ? (int)(n - n0) * q.image + (ih * p.Wlim + iw) * 4 : (int)0x80000000;
  }
  float reg[IT][8];
  auto fetch = [&](const int chunk) __attribute__((always_inline)) {
    const int c0 = chunk * kBK + 8 * half;
#pragma unroll
    for (int it = 0; it < IT; ++it)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int vo = c0 + e < q.C ? voff[it] : (int)0x80000000;
        reg[it][e] = as_float(__builtin_amdgcn_raw_buffer_load_b32(srd, vo, (c0 + e) * q.plane, 0));
      }
  };
  const float lift = q.w ? kLift : 1.f;
  auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
#pragma unroll
      for (int e = 0; e < 8; ++e) reg[it][e] *= lift;
      uintx4 t[kTerms];
      split8(reg[it], t);
      if (it * 128 + pp0 < k.px) {
#pragma unroll
        for (int i = 0; i < kTerms; ++i) *reinterpret_cast<uintx4*>(lds + at + it * 128 * kUnit + 16 * i) = t[i];
      }
    }
  };

  // Products of the first terms in `acc`, all others, 2^-8 of them and less, in `small`: the long chain has one
  // rounding per sixteen channels and tap where a single one would have six.
  floatx16 acc[1][NT], small[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][y][r] = small[y][r] = 0.f;

  int base[NT];   // the lane's pixels in the patch
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    const int m = m0 + (wn * NT + y) * 32 + l32;
    uint32_t n;
    base[y] = (int)(virtual_pixel((uint32_t)(m < k.M ? m : m0), n) - first + (uint32_t)(h * k.px)) * kUnit;
  }

  // the wave's weights: one run of 3 KB per tap, fetched two taps ahead into the registers that a tap is done with
  const uintx4* wptr = q.wt + k.wt + ((size_t)(i0 / 32 + wm) * q.chunks + q0) * (size_t)(k.taps * kTerms * 64);
  uintx4 w1[kTerms], w2[kTerms];
  auto load_weights = [&](uintx4 (&to)[kTerms]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kTerms; ++i) to[i] = wptr[i * 64 + lane];
    wptr += kTerms * 64;
  };
  uintx4 b[2][2][kTerms];   // two 32-pixel tiles at a time, and the two behind them
  auto load_pixels = [&](const int y, const int offset, uintx4 (&to)[2][kTerms]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < kTerms; ++i) to[j][i] = *reinterpret_cast<const uintx4*>(lds + base[y + j] + offset + 16 * i);
  };
  // One tap: 6*NT matrix instructions.  b[first_buf] holds its first pixels; a step's pixels are read while the step
  // before it multiplies, and two tiles' products alternate, since each waits for the one before it on the same
  // accumulator.  The weights that are read past a wave's last tap are not used.
  auto tap = [&](uintx4 (&w)[kTerms], const int first_buf, const int off, const int next) __attribute__((always_inline)) {
    bf16x8 a[kTerms];
#pragma unroll
    for (int i = 0; i < kTerms; ++i) a[i] = __builtin_bit_cast(bf16x8, w[i]);
#pragma unroll
    for (int y = 0; y < NT; y += 2) {
      auto& x = b[(first_buf + y / 2) & 1];
      auto& behind = b[(first_buf + y / 2 + 1) & 1];
      if (y + 2 < NT) load_pixels(y + 2, off, behind);
      else load_pixels(0, next, behind);
      __builtin_amdgcn_sched_barrier(0);
      auto product = [&](const int i, const int term, floatx16 (&to)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          to[y + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], __builtin_bit_cast(bf16x8, x[j][term]), to[y + j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      };
      product(0, 2, small);
      product(0, 0, acc[0]);
      product(2, 0, small);
      product(1, 1, small);
      product(0, 1, small);
      product(1, 0, small);
    }
    load_weights(w);
    __builtin_amdgcn_sched_barrier(0);
  };

  const bool whole = q.partial == nullptr;
  if constexpr (EPI) {
    if (whole && p.epi.on) epilogue_constants<BM>(p, 0, i0, tid, epi_lds);   // published by the barrier below
  }
  fetch(q0);
  load_weights(w1);
  load_weights(w2);
  stage();
  __syncthreads();
  load_pixels(0, 0, b[0]);
  if (q0 + 1 < q1) fetch(q0 + 1);   // in flight across this chunk's matrix instructions
  // The taps of all chunks in pairs, whatever their number.  One too many has zero weights.
  int c = q0, t = 0, ts = 0, row = 0, off = 0, next = 0;   // tap t of chunk c, column ts of its kernel row
  auto look = [&]() __attribute__((always_inline)) {   // where the tap behind this one lies
    next = off + k.tapCol;
    if (++ts == k.S) {
      ts = 0;
      next = row += k.tapRow;
    }
    if (t + 1 == k.taps) next = 0;
  };
  auto advance = [&](const int next_buf) __attribute__((always_inline)) {
    off = next;
    if (++t == k.taps) {
      t = ts = row = 0;
      if (++c < q1) {
        __syncthreads();   // the patch has been read by every wave
        stage();
        __syncthreads();
        load_pixels(0, 0, b[next_buf]);
        if (c + 1 < q1) fetch(c + 1);
      }
    }
    look();
  };
  look();
  const int total = (q1 - q0) * k.taps;
  constexpr int kOdd = (NT / 2) & 1;   // the buffer that a pair's second tap begins with
  for (int i = 0; i < total; i += 2) {
    tap(w1, 0, off, next);
    advance(kOdd);
    if (i + 1 == total)
#pragma unroll
      for (int j = 0; j < kTerms; ++j) w2[j] = uintx4{0, 0, 0, 0};
    tap(w2, kOdd, off, next);
    advance(0);
  }
  int again = lane;
  asm("" : "+v"(again));   // where a lane's values lie is worked out again: kept over the loop it would take registers there
  const int col = again & 31, hh = again >> 5;
  uint32_t obase[NT];
  bool mok[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    const int m = m0 + (wn * NT + y) * 32 + col;
    mok[y] = m < k.M;
    uint32_t n, u, v;
    split_pixel(mok[y] ? (uint32_t)m : 0u, n, u, v);
    obase[y] = n * (uint32_t)p.outStrideN + (u * (uint32_t)p.ou + (uint32_t)k.ouh) * (uint32_t)p.outRow + v * (uint32_t)p.ov + (uint32_t)k.ovw;
  }
#pragma unroll
  for (int y = 0; y < NT; ++y) acc[0][y] += small[y];

  if (q.w) {
    if (__builtin_amdgcn_ballot_w64(not_finite<1, NT>(acc))) {   // sums that three terms do not hold
      WaveOperands<1, NT> o;
      o.R = k.taps / k.S; o.S = k.S; o.wC = q.wC; o.wRow = k.wRow; o.wCol = k.wCol; o.dh = k.dh; o.dw = k.dw;
      o.H = p.Hlim; o.W = p.Wlim; o.srcRow = p.Wlim; o.plane = q.plane / 4;
      o.w[0] = q.w + (long long)min(i0 + wm * 32 + col, p.I - 1) * q.wI + k.w0;
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        uint32_t n, u, v;
        split_pixel((uint32_t)min(m0 + (wn * NT + y) * 32 + col, k.M - 1), n, u, v);
        o.src[y] = (const float*)((const char*)q.src + (long long)n * q.image);
        o.ih[y] = (int)u + k.bh;
        o.iw[y] = (int)v + k.bw;
      }
      float32_sums<1, NT>(acc, o, q0 * kBK, min(q.C, q1 * kBK), hh);
    } else {
#pragma unroll
      for (int y = 0; y < NT; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][y][r] *= kLower;
    }
  }
  if constexpr (EPI) {
    if (whole && p.epi.on) {
#pragma unroll
      for (int y = 0; y < NT; y += 2) {   // two tiles at a time: their residuals and masks are as many registers again
        const floatx16 two[1][2] = {{acc[0][y], acc[0][y + 1]}};
        const uint32_t ob[2] = {obase[y], obase[y + 1]};
        const bool ok[2] = {mok[y], mok[y + 1]};
        store_through_epilogue<BM, 1, 2>(p, two, ob, ok, i0, wm * 32, hh, epi_lds);
      }
    }
  }
  // accumulator register r of a 32x32 tile holds row 8*(r/4) + 4*h + r%4, column l32
  float* out = whole ? p.out : q.partial + (size_t)blockIdx.z * (size_t)q.outElems;
  if (!EPI || !whole || !p.epi.on) {
    const bool biased = whole && p.bias != nullptr;
    const uint32_t hoff = (uint32_t)(4 * hh * p.outStrideI);
    const int srow = __builtin_amdgcn_readfirstlane(i0 + wm * 32);
    float bz[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bz[r] = biased ? p.bias[min(srow + 8 * (r >> 2) + 4 * hh + (r & 3), p.I - 1)] : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // every load done before the first store: they share one counter
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = srow + 8 * (r >> 2) + (r & 3);
      float* __restrict__ rowp = out + (size_t)row * (size_t)p.outStrideI;
      if (row + 4 * hh < p.I) {
#pragma unroll
        for (int y = 0; y < NT; ++y)
          if (mok[y]) rowp[obase[y] + hoff] = biased ? acc[0][y][r] + bz[r] : acc[0][y][r];
      }
    }
  }
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
size_t align_up(size_t v) { return (v + 255) / 256 * 256; }

struct Plan {
  int WM, NT, IT, Ipad, maxPx, chunks, perSplit, splits, tiles;
  int px[kPatchClasses], PW[kPatchClasses], VR[kPatchClasses], block0[kPatchClasses];
  size_t at[kPatchClasses], wt, partial;   // the classes' weights (units of 16 bytes); bytes of workspace
  double cost, longest;   // microseconds: of the launch, of its longest block
};

int g_patch = 1;   // tests: 0 = never, 2 = wherever they can

// The virtual image's rows per image, or its pitch: what the taps reach, less the zeros that two frames share.
int framed(int pixels, int taps, int dil, int pad, int limit) {
  const int reach = (taps - 1) * dil, behind = pixels - 1 + reach - pad - (limit - 1);
  return pixels + reach - std::max(0, std::min({pad, behind, reach}));
}

bool make_plan(const PatchConv& c, Plan* best) {
  best->cost = -1;
  for (const auto& shape : {std::pair{4, 4}, {2, 4}, {2, 2}}) {
    Plan pl{};
    pl.WM = shape.first; pl.NT = shape.second;
    const int BM = 32 * pl.WM, BN = 128 * pl.NT / pl.WM;
    pl.Ipad = ceil_div(c.I, BM) * BM;
    pl.chunks = ceil_div(c.C, kBK);
    size_t wt = 0;
    bool fits = true;
    for (int k = 0; k < c.n && fits; ++k) {
      const PatchConvClass& g = c.c[k];
      const long long M = (long long)c.N * g.U * g.V;
      pl.VR[k] = framed(g.U, g.R, g.dh, g.ph, c.H);
      pl.PW[k] = framed(g.V, g.S, g.dw, g.pw, c.W);
      // the longest range of the virtual image that BN consecutive pixels and their taps cover
      const long long rows = (BN + g.V - 2) / g.V, images = (BN + (long long)g.U * g.V - 2) / ((long long)g.U * g.V);
      const long long px = BN + rows * (pl.PW[k] - g.V) + images * (long long)(pl.VR[k] - g.U) * pl.PW[k] +
                           (long long)(g.R - 1) * g.dh * pl.PW[k] + (long long)(g.S - 1) * g.dw;
      fits = px <= 512;
      pl.px[k] = (int)px;
      pl.maxPx = std::max(pl.maxPx, pl.px[k]);
      pl.block0[k] = pl.tiles;
      pl.tiles += (pl.Ipad / BM) * ceil_div(M, BN);
      pl.at[k] = wt;
      wt += (size_t)pl.Ipad / 32 * pl.chunks * g.R * g.S * kTerms * 64;
    }
    if (!fits) continue;
    pl.IT = pl.maxPx <= 384 ? 3 : 4;
    pl.wt = align_up((wt + kReadPast * kTerms * 64) * 16);
    // Microseconds, fitted to 75 launches of 4 to 2000 blocks (10 % root mean square): a chunk of a block that
    // shares its compute unit, a block's start and end; a block that has the unit for itself takes a sixth longer.
    // Shares of a reduction are written, read and added.  (The weights' layout costs the same for all.)
    for (int s = 1; s <= 8 && s <= pl.chunks; ++s) {
      const int per = ceil_div(pl.chunks, s);
      if (ceil_div(pl.chunks, per) != s) continue;
      double work = 0, longest = 0, outputs = 0;
      for (int k = 0; k < c.n; ++k) {
        const int taps = c.c[k].R * c.c[k].S;
        const double block = per * (pl.NT == 4 ? 0.55 * taps + 1.0 : 0.32 * taps + 1.0) + 4;
        work += block * s * ((k + 1 < c.n ? pl.block0[k + 1] : pl.tiles) - pl.block0[k]);
        longest = std::max(longest, block);
        outputs += (double)c.I * c.N * c.c[k].U * c.c[k].V;
      }
      const double cost = std::max(1.17 * longest, work / tt::compute_units() + 0.1 * longest) + (s > 1 ? 5 + (2 * s + 1) * 4e-6 / 7 * outputs : 0);
      if (best->cost < 0 || cost < best->cost) {
        pl.perSplit = per;
        pl.splits = s;
        pl.cost = cost;
        pl.longest = longest;
        pl.partial = s > 1 ? align_up(sizeof(float) * (size_t)s * (size_t)outputs) : 0;
        *best = pl;
      }
    }
  }
  return best->cost >= 0;
}

}  // namespace

namespace ttc {

size_t patch_workspace(const PatchConv& c) {
  Plan pl;
  return make_plan(c, &pl) ? pl.wt + pl.partial : 0;
}

bool patch_conv_takes(const PatchConv& c, bool f32) {
  if (g_patch == 0 || c.n < 1 || c.taps > kMaxTaps) return false;
  double sums = 0;
  for (int k = 0; k < c.n; ++k) {
    const PatchConvClass& g = c.c[k];
    if ((g.R - 1LL) * g.dh > 512 || (g.S - 1LL) * g.dw > 512) return false;   // wider than a patch
    sums += (double)g.R * g.S * g.U * g.V;
  }
  // most calls are too small: no plan for them (0.1 to 0.2 us of host time each)
  const double gigas = 2e-9 * c.I * c.C * c.N * sums;
  if (g_patch != 2 && (c.taps < 4 || gigas < (f32 ? 4.0 : 1.5))) return false;
  Plan pl;
  if (!make_plan(c, &pl)) return false;
  // 32-bit offsets: virtual pixels of the batch, source bytes of the images that a patch touches
  const long long image = 4LL * c.C * c.H * c.W;
  for (int k = 0; k < c.n; ++k) {
    const long long frame = (long long)pl.VR[k] * pl.PW[k];
    if ((c.N + 1) * frame + 1024 >= (1LL << 31) || (pl.px[k] / frame + 2) * image >= (1LL << 31)) return false;
  }
  if (pl.Ipad / 32 > 65535) return false;   // the grid of patch_weights
  if (g_patch == 2) return true;
  if (pl.wt + pl.partial > ((size_t)1 << 30)) return false;   // workspace stays with the library
  // Against the kernels that gather in place, whose time is about 16 us and 7 us per 1e9 products and sums (53
  // launches of 0.5 to 25e9; they take less where a long reduction is shared between many blocks, and more, up to
  // twice, where it is not).  So it is taken for 28 of 75 launches, 1.12 times as fast on average: 64 channels
  // 32x32 at batch 128 72.1 us, 62.7 here; 128 channels 16x16 98.0, 67.2; 256 channels 8x8 77.0, 70.4; 160 to 192
  // channels 45x37 at batch 24 183.9, 117.0; and not for 128 channels 28x28 at batch 8 (29.3, 32.9) or 3 channels
  // (23.4, 56.8), whose rows and channels are mostly padding.
  // In float32 arithmetic small calls, which gain a few microseconds at most, stay with them, and the line lies a little
  // higher: it was fitted to float32 instructions (94 us for 9.7e9 and 119 to 138 for 14.8e9, where these take 63 to 68
  // and 90 to 102).  From 4e9 on the kernels that gather run on three terms too (f32_terms); 7.0 here moves some
  // launches of a PreAct-ResNet-18 step and its time by less than runs differ (4.70 ms, 4.73).
  const double padding = (double)pl.chunks * kBK * pl.Ipad / ((double)c.C * c.I);
  const double weights = 4e-6 * c.I * c.C * c.taps;
  if (padding > 1.5 || pl.cost + 3 + weights >= 16 + (f32 ? 7.5 : 7.0) * gigas) return false;
  if (f32) return true;
  // Outside float32 arithmetic, where the other side is the same product, one in eight of 1339 launches that are left was
  // more than 8 % slower here (194.9 ms here, 223.7 there, 191.6 at best).  Most had between one and two blocks to a compute
  // unit, of which some run two while the others wait, or several classes; and the others' time grows with the padding of
  // their rows.  With these three in the line 1045 stay (193.4 ms, 32 slower by more than 8 %; of another draw 3424, 3.6 %
  // of them slower, 1.18 times as fast in all): 36 to 363 channels 4x4 7x28 at batch 24 41.9 us and 31.7 go back, 96 to 62
  // 5x5 7x42 at batch 58 65.4 and 54.7.
  const int blocks = pl.tiles * pl.splits, cus = tt::compute_units();
  const double here = blocks > cus && blocks <= 2 * cus ? std::max(pl.cost, 1.75 * pl.longest) : pl.cost;
  const int rows = c.I > 64 ? 128 : 32;
  return here + weights + (c.n > 1 ? 6 : 0) < 14 + (2.3 + 4.7 * (ceil_div(c.I, rows) * rows) / c.I) * gigas;
}

int patch_conv_launch(const PatchConv& c, const float* x, const float* w, const float* bias, float* out, const Epilogue* epi,
                      bool f32, int prof_id, int* plan8) {
  Plan pl;
  if (!make_plan(c, &pl)) return tt::fail(-1, "patch convolution: no plan");
  void* ws = nullptr;
  if (tt::workspace(pl.wt + pl.partial, &ws)) return -1;
  hipStream_t st = tt::stream();
  Igemm p{};
  p.bias = bias; p.out = out;
  if (epi) p.epi = *epi;
  p.I = c.I; p.Ipad = pl.Ipad; p.M = c.N * c.outPlane;
  p.divUV = tt::make_fastdiv((uint32_t)c.outPlane);
  p.Hlim = c.H; p.Wlim = c.W;
  p.outStrideN = c.I * c.outPlane; p.outStrideI = c.outPlane; p.outRow = c.outRow;
  p.ou = c.ou; p.ov = c.ov;
  Patch q{};
  q.src = x; q.wt = (const uintx4*)ws;
  q.partial = pl.splits > 1 ? (float*)((char*)ws + pl.wt) : nullptr;
  q.outElems = (long long)p.I * p.M;
  q.C = c.C; q.chunks = pl.chunks; q.perSplit = pl.perSplit;
  q.plane = 4 * c.H * c.W; q.image = q.plane * c.C;
  q.maxPx = pl.maxPx; q.images = c.N;
  if (f32) {
    q.w = w;
    q.wI = c.dgrad ? c.taps : c.C * c.taps;
    q.wC = c.dgrad ? c.I * c.taps : c.taps;
  }
  q.classes = c.n;
  PatchTaps taps{};
  taps.n = c.n;
  for (int k = 0; k < c.n; ++k) {
    const PatchConvClass& g = c.c[k];
    q.c[k] = PatchClass{c.N * g.U * g.V, tt::make_fastdiv((uint32_t)(g.U * g.V)), tt::make_fastdiv((uint32_t)g.V), -g.ph, -g.pw, g.ouh, g.ovw,
                        g.R * g.S, g.S, pl.PW[k], pl.VR[k], tt::make_fastdiv((uint32_t)pl.PW[k]), tt::make_fastdiv((uint32_t)pl.VR[k]),
                        pl.px[k], g.dh * pl.PW[k] * kUnit, g.dw * kUnit, g.dh, g.dw, g.w0, g.wRow, g.wCol, pl.block0[k], pl.at[k]};
    taps.taps[k] = g.R * g.S; taps.S[k] = g.S;
    taps.w0[k] = g.w0; taps.wRow[k] = g.wRow; taps.wCol[k] = g.wCol; taps.wt[k] = pl.at[k];
  }
  {
    tt::ProfScope prof(TT_PROF_CONV_PREP);
    const int run = (c.dgrad ? 32 : kBK) * c.taps, outer = c.dgrad ? kBK : 32;
    const dim3 grid((unsigned)pl.chunks, (unsigned)(pl.Ipad / 32));
    const size_t lds = sizeof(float) * (size_t)outer * (run + 1);
    const tt::FastDiv divRun = tt::make_fastdiv((uint32_t)run);
    if (c.dgrad) patch_weights<true><<<grid, kThreads, lds, st>>>(w, (uintx4*)ws, c.I, c.C, c.taps, divRun, pl.chunks, f32 ? kLift : 1.f, taps);
    else patch_weights<false><<<grid, kThreads, lds, st>>>(w, (uintx4*)ws, c.I, c.C, c.taps, divRun, pl.chunks, f32 ? kLift : 1.f, taps);
    TT_LAUNCH_CHECK();
  }
  const int BM = 32 * pl.WM, BN = 128 * pl.NT / pl.WM;
  const int plan[8] = {BM, BN, pl.tiles, pl.Ipad / BM, -4, pl.tiles, pl.splits, kModeTapMask | 3 << 8};
  std::copy(plan, plan + 8, plan8);
  tt::ProfScope prof(prof_id);
  const dim3 grid((unsigned)pl.tiles, 1, (unsigned)pl.splits);
  const size_t lds = 2 * (size_t)pl.maxPx * kUnit + 4 * sizeof(float) * BM;
  const bool epilogue = p.epi.on && pl.splits == 1;
#define TT_PATCH(WM, NT, IT)                                                     \
  (epilogue ? patch_product<WM, NT, IT, true><<<grid, kThreads, lds, st>>>(p, q) \
            : patch_product<WM, NT, IT, false><<<grid, kThreads, lds, st>>>(p, q))
  if (pl.WM == 4) {
    if (pl.IT == 3) TT_PATCH(4, 4, 3); else TT_PATCH(4, 4, 4);
  } else if (pl.NT == 4) {
    if (pl.IT == 3) TT_PATCH(2, 4, 3); else TT_PATCH(2, 4, 4);
  } else {
    if (pl.IT == 3) TT_PATCH(2, 2, 3); else TT_PATCH(2, 2, 4);
  }
#undef TT_PATCH
  TT_LAUNCH_CHECK();
  if (pl.splits > 1) return add_partials(p, q.partial, pl.splits);
  return 0;
}

}  // namespace ttc

extern "C" int tt_conv2d_patch_enable(int on) {
  TT_API_LOCK();
  TT_REQUIRE(on >= 0 && on <= 2, "tt_conv2d_patch_enable: %d is out of range (0..2)", on);
  g_patch = on;
  return 0;
}
