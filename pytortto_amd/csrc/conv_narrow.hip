// Convolutions with few rows: forward passes of a group with up to 16 output channels, input gradients of
// up to 16 input channels, and weight gradients with few rows or columns (depthwise and grouped layers, layers in
// front of or behind an image).
//
// The matrix instructions compute 32 rows whatever a layer has, so these layers run on the vector unit instead:
// a thread owns pixels, keeps all rows of them in registers and reads a gathered value once for all
// rows.  Whether a tap lies inside the image, and where, is worked out once for four or eight channels, which
// only move the scalar offset of a buffer load.  Weights lie in LDS, [step][row], and every lane reads the
// same 16 bytes (a broadcast).  Bound by the vector unit, and with long reductions by the passage of a load per
// value through the address unit.  Channels in runs of eight, all taps of a run after each other: with whole taps
// outermost a block's values left the L1, and the L2, between taps (64 channels to 3, 4x4 at stride 2, 128 images of
// 64x64: 198 us, 86 in runs).
// Sums: four or eight products are added on their own, then to those of 128 steps, then to the rest: shorter
// chains than the matrix instructions' one over the whole reduction, and a smaller error in all of 90 cases.
// Grouped 4 to 16 channels, 3x2, 128 images of 64x64 (a reference notebook's layer), forward, input and weight gradient:
// 18.2 us, 29.1 and 50.8 with the matrix kernels, 11.5, 18.4 and 19.9 here, and no launches for weights (7.2) or to clear (5.2).
#include <algorithm>
#include <type_traits>

#include "conv_narrow.h"

namespace {

using namespace ttc;

constexpr int kSteps = 128;   // steps (tap, channel) of the weights in LDS at a time

__device__ __forceinline__ float rounded_bf16(float v) { return (float)(__bf16)v; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t srd_of(const float* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, kSrdRecords, kSrdFlags);
}

// KT rows (I <= KT), PX pixels per thread; BF: operands rounded to bfloat16; FEW: fewer than four channels, so
// that four taps are fetched together instead of four channels.
// EPI: the launch applies NarrowConv::epi to what it stores, with the operations of the matrix kernels' epilogue in their order.
template <int KT, int PX, bool BF, bool FEW, bool EPI>
__global__ __launch_bounds__(kThreads) void conv_narrow(const NarrowConv p) {
  constexpr int kAhead = PX == 1 ? 8 : 4;
  __shared__ __align__(16) float ws[kSteps][KT];
  __shared__ float consts[EPI ? 4 * KT : 1];   // per row: mean, gamma / sd, beta, bias
  int ci = 0;
  while (ci + 1 < p.n && (int)blockIdx.x >= p.c[ci + 1].block0) ++ci;
  const NarrowClass& c = p.c[ci];
  const int g = blockIdx.y, t = threadIdx.x;
  const int m0 = ((int)blockIdx.x - c.block0) * (kThreads * PX);
  const int n0 = (int)tt::fd_div((uint32_t)m0, c.divUV);
  const __amdgpu_buffer_rsrc_t src = srd_of(p.src + (size_t)n0 * p.srcN + (size_t)g * p.srcG);
  int ih0[PX], iw0[PX], nb[PX];
  float acc[PX][KT] = {};
#pragma unroll
  for (int x = 0; x < PX; ++x) {
    const int m = m0 + t + x * kThreads;
    const uint32_t mm = (uint32_t)min(m, c.M - 1);
    const uint32_t n = tt::fd_div(mm, c.divUV), rem = mm - n * c.divUV.d;
    const uint32_t u = tt::fd_div(rem, c.divV), v = rem - u * c.divV.d;
    ih0[x] = m < c.M ? (int)u * p.su + c.bh : kInvalid;   // pixels past the end read nothing
    iw0[x] = (int)v * p.sv + c.bw;
    nb[x] = ((int)n - n0) * p.srcN;
  }
  // byte offset of tap (b, cc) for pixel x; bit 31 where it lies outside, which reads 0
  auto at = [&](int x, int b, int cc) __attribute__((always_inline)) {
    const int ih = ih0[x] + b * p.stepH, iw = iw0[x] + cc * p.stepW;
    const bool ok = (unsigned)ih < (unsigned)p.Hlim && (unsigned)iw < (unsigned)p.Wlim;
    return ok ? 4u * (uint32_t)(nb[x] + ih * p.Wlim + iw) : 0x80000000u;
  };
  auto value = [&](uint32_t off, int channel) __attribute__((always_inline)) {
    const float v = as_float(__builtin_amdgcn_raw_buffer_load_b32(src, (int)off, 4 * channel * p.plane, 0));
    return BF ? rounded_bf16(v) : v;
  };
  if constexpr (EPI) {
    if (t < KT) {
      const int ch = g * p.I + min(t, p.I - 1);
      float m = 0.f, k1 = 1.f, k0 = -0.f;   // leave a value as it is
      if (p.epi.norm) {
        m = p.epi.mean[ch];
        k1 = __fdiv_rn(p.epi.gamma ? p.epi.gamma[ch] : 1.0f, __fsqrt_rn(__fadd_rn(p.epi.var[ch], p.epi.eps)));
        k0 = p.epi.beta ? p.epi.beta[ch] : 0.0f;
      }
      consts[t] = m;
      consts[KT + t] = k1;
      consts[2 * KT + t] = k0;
      consts[3 * KT + t] = p.bias ? p.bias[ch] : -0.f;
    }
  }
  const int taps = c.TB * c.TC;
  // The reduction runs over units: four taps of one channel after the other (FEW: all channels of four
  // taps), or kAhead channels of a tap, channels outermost, so that a block's values stay in the L1 over the taps.
  const int chunks = FEW ? 1 : (p.A + kAhead - 1) / kAhead;
  const int units = FEW ? (taps + 3) / 4 : chunks * taps, unit_steps = FEW ? 4 * p.A : kAhead;
  const int stage = kSteps / unit_steps;
  // what unit u's k-th step is: tap, channel; nothing beyond `count`
  auto unit = [&](int u, int& tap, int& channel, int& count) __attribute__((always_inline)) {
    if constexpr (FEW) {
      tap = 4 * u;
      channel = 0;
      count = min(4, taps - tap);
    } else {
      const int chunk = (int)tt::fd_div((uint32_t)u, c.divTaps);
      tap = u - chunk * taps;
      channel = chunk * kAhead;
      count = min(kAhead, p.A - channel);
    }
  };
  float in[2][FEW ? 1 : kAhead][PX];   // values of a unit, fetched while the one in front of it is multiplied
  auto fetch = [&](int set, int u) __attribute__((always_inline)) {
    int tap, channel, count;
    unit(u, tap, channel, count);
    const int b = (int)tt::fd_div((uint32_t)tap, c.divTC), cc = tap - b * c.TC;
    uint32_t off[PX];
#pragma unroll
    for (int x = 0; x < PX; ++x) off[x] = at(x, b, cc);
#pragma unroll
    for (int k = 0; k < (FEW ? 1 : kAhead); ++k)
#pragma unroll
      for (int x = 0; x < PX; ++x) in[set][k][x] = value(off[x], channel + min(k, count - 1));
  };
  if constexpr (!FEW) {
    if (units > 0) fetch(0, 0);
  }
  for (int u0 = 0; u0 < units; u0 += stage) {
    const int here = min(stage, units - u0);
    __syncthreads();
    for (int e = t; e < here * unit_steps * KT; e += kThreads) {
      const int i = e % KT, step = e / KT;
      const int u = FEW ? (int)tt::fd_div((uint32_t)step, p.divUnit) : step / kAhead, k = step - u * unit_steps;
      int tap, channel, count;
      unit(u0 + u, tap, channel, count);
      if constexpr (FEW) {   // [tap][channel]
        const int ahead = (int)tt::fd_div((uint32_t)k, p.divA);
        tap += ahead;
        channel = k - ahead * p.A;
      } else {
        channel += k;
      }
      const int b = (int)tt::fd_div((uint32_t)tap, c.divTC), cc = tap - b * c.TC;
      float v = 0.f;
      if (i < p.I && tap < taps && channel < p.A)
        v = p.w[(size_t)g * p.wG + (size_t)i * p.wI + (size_t)channel * p.wA + (size_t)((c.r0 + b * p.rs) * p.S + c.s0 + cc * p.ss)];
      ws[step][i] = BF ? rounded_bf16(v) : v;
    }
    __syncthreads();
    float part[PX][KT] = {};
    // products of the first n of kN steps, `stride` apart in LDS: added up on their own first
    auto add = [&](auto steps, int s, int stride, const auto& from, int n) __attribute__((always_inline)) {
      constexpr int kN = decltype(steps)::value;
#pragma unroll
      for (int q = 0; q < KT / 4; ++q) {
        float sum[PX][4];
#pragma unroll
        for (int k = 0; k < kN; ++k) {
          if (k > 0 && k >= n) break;
          const floatx4 w4 = *reinterpret_cast<const floatx4*>(&ws[s + k * stride][4 * q]);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int x = 0; x < PX; ++x) sum[x][j] = k == 0 ? from[k][x] * w4[j] : fmaf(from[k][x], w4[j], sum[x][j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int x = 0; x < PX; ++x) part[x][4 * q + j] += sum[x][j];
      }
    };
    if constexpr (FEW) {
      for (int u = 0; u < here; ++u) {
        const int tap = 4 * (u0 + u), count = min(4, taps - tap);
        uint32_t off[4][PX];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int b = (int)tt::fd_div((uint32_t)(tap + k), c.divTC), cc = tap + k - b * c.TC;
#pragma unroll
          for (int x = 0; x < PX; ++x) off[k][x] = k < count ? at(x, b, cc) : 0x80000000u;
        }
        for (int a = 0; a < p.A; ++a) {
          float four[4][PX];
#pragma unroll
          for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int x = 0; x < PX; ++x) four[k][x] = value(off[k][x], a);
          if (count == 4) add(std::integral_constant<int, 4>{}, u * unit_steps + a, p.A, four, 4);
          else add(std::integral_constant<int, 4>{}, u * unit_steps + a, p.A, four, count);
        }
      }
    } else {
      for (int j = 0; j < here; j += 2) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int u = u0 + j + half;   // (stages are of even length: set `half` holds unit u)
          if (j + half >= here) break;
          if (u + 1 < units) fetch(1 - half, u + 1);
          int tap, channel, count;
          unit(u, tap, channel, count);
          if (count == kAhead) add(std::integral_constant<int, kAhead>{}, (j + half) * kAhead, 1, in[half], kAhead);
          else add(std::integral_constant<int, kAhead>{}, (j + half) * kAhead, 1, in[half], count);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < PX; ++x)
#pragma unroll
      for (int i = 0; i < KT; ++i) acc[x][i] += part[x][i];
  }
  if constexpr (EPI) __syncthreads();   // (a class without taps has met no barrier yet)
#pragma unroll
  for (int x = 0; x < PX; ++x) {
    const int m = m0 + t + x * kThreads;
    if (m >= c.M) continue;
    const uint32_t n = tt::fd_div((uint32_t)m, c.divUV), rem = (uint32_t)m - n * c.divUV.d;
    const uint32_t u = tt::fd_div(rem, c.divV), v = rem - u * c.divV.d;
    const size_t at0 = (size_t)n * p.outN + (size_t)g * p.outG + (size_t)(((int)u * p.ou + c.ouh) * p.outRow + (int)v * p.ov + c.ovw);
    if constexpr (EPI) {
      const float floor_ = p.epi.relu ? 0.f : -__builtin_huge_valf();
      float rs[KT], ms[KT];
#pragma unroll
      for (int i = 0; i < KT; ++i) {
        const size_t e = at0 + (size_t)min(i, p.I - 1) * p.outI;
        rs[i] = p.epi.res ? p.epi.res[e] : -0.f;
        ms[i] = p.epi.mask ? p.epi.mask[e] : 1.f;
      }
#pragma unroll
      for (int i = 0; i < KT; ++i)
        if (i < p.I) {
          float o = acc[x][i] + consts[3 * KT + i];
          o = fmaf(o - consts[i], consts[KT + i], consts[2 * KT + i]) + rs[i];
          o = (o > floor_ || o != o) ? o : floor_;
          p.out[at0 + (size_t)i * p.outI] = o * (ms[i] > 0.f ? 1.f : 0.f);
        }
    } else {
#pragma unroll
      for (int i = 0; i < KT; ++i)
        if (i < p.I) p.out[at0 + (size_t)i * p.outI] = p.bias ? acc[x][i] + p.bias[g * p.I + i] : acc[x][i];
    }
  }
}

// ---- weight gradient ---------------------------------------------------------------------------------
// A block owns a KT x JT piece of one group's dw and a run of output pixels; a thread forms the outer product of
// KT values of dy and JT of x for every pixel of its own, so a fetched value serves KT or JT products.
// Threads' sums are added across lanes, waves (float64) and, by narrow_sum, blocks (float64).

__device__ __forceinline__ float lanes_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));    // lane ^ 1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));    // lane ^ 2
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));   // half rows
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));   // rows of 16
  v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401f));                      // lane ^ 16
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)) + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
}

template <int KT, int JT, bool BF>
__global__ __launch_bounds__(kThreads) void wgrad_narrow(const NarrowWgrad p) {
  __shared__ float sums[4][KT * JT];
  const int t = threadIdx.x, g = blockIdx.y, split = blockIdx.z;
  const int it = (int)blockIdx.x % p.tilesI, jt = (int)blockIdx.x / p.tilesI;
  // columns: byte offset of (channel, tap) behind a window's first element, and tap number (uniform)
  int joff[JT], jtap[JT], ioff[KT];
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    const uint32_t col = (uint32_t)min(jt * JT + j, p.J - 1);   // columns past the end: never stored
    const uint32_t ch = tt::fd_div(col, p.divRS), rs = col - ch * p.divRS.d;
    const uint32_t r = tt::fd_div(rs, p.divS), s = rs - r * p.divS.d;
    joff[j] = __builtin_amdgcn_readfirstlane(4 * ((int)ch * p.HW + (int)r * p.dh * p.W + (int)s * p.dw));
    jtap[j] = __builtin_amdgcn_readfirstlane((int)rs);
  }
#pragma unroll
  for (int i = 0; i < KT; ++i) ioff[i] = __builtin_amdgcn_readfirstlane(4 * min(it * KT + i, p.Kg - 1) * p.PQ);
  float acc[KT][JT] = {};
  const int from = split * p.perSplit, to = min(p.M, from + p.perSplit);
  for (int base = from; base < to; base += kThreads) {
    const int n0 = (int)tt::fd_div((uint32_t)base, p.divPQ);
    const __amdgpu_buffer_rsrc_t dy = srd_of(p.dy + (size_t)n0 * p.dyN + (size_t)g * p.dyG);
    const __amdgpu_buffer_rsrc_t xs = srd_of(p.x + ((long long)n0 * p.xN + (long long)g * p.xG - p.xBias));
    const int m = base + t;
    const uint32_t mm = (uint32_t)min(m, to - 1);
    const uint32_t n = tt::fd_div(mm, p.divPQ), pq = mm - n * p.divPQ.d;
    const uint32_t u = tt::fd_div(pq, p.divQ), v = pq - u * p.divQ.d;
    const int ih = (int)u * p.sh - p.ph, iw = (int)v * p.sw - p.pw;
    const uint32_t xo = 4u * (uint32_t)(((int)n - n0) * p.xN + ih * p.W + iw + p.xBias);
    const uint32_t yo = m < to ? 4u * (uint32_t)(((int)n - n0) * p.dyN + (int)pq) : 0x80000000u;   // pixels past the end: dy reads 0 ...
    uint32_t cols = 0, inside = 0;                                                                 // ... and so does x
    for (int s = 0; s < p.S; ++s) cols |= (uint32_t)((unsigned)(iw + s * p.dw) < (unsigned)p.W) << s;
    for (int r = 0; r < p.R; ++r)
      if ((unsigned)(ih + r * p.dh) < (unsigned)p.H) inside |= cols << (r * p.S);
    const uint32_t outside = m < to ? ~inside : ~0u;
    float a[KT], b[JT];
#pragma unroll
    for (int i = 0; i < KT; ++i) a[i] = as_float(__builtin_amdgcn_raw_buffer_load_b32(dy, (int)yo, ioff[i], 0));
#pragma unroll
    for (int j = 0; j < JT; ++j)
      b[j] = as_float(__builtin_amdgcn_raw_buffer_load_b32(xs, (int)(((outside >> jtap[j]) << 31) | xo), joff[j], 0));
    if constexpr (BF) {
#pragma unroll
      for (int i = 0; i < KT; ++i) a[i] = rounded_bf16(a[i]);
#pragma unroll
      for (int j = 0; j < JT; ++j) b[j] = rounded_bf16(b[j]);
    }
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
      for (int j = 0; j < JT; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
  }
  const int lane = t & 63, wave = t >> 6;
#pragma unroll
  for (int i = 0; i < KT; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const float s = lanes_sum(acc[i][j]);
      if (lane == 0) sums[wave][i * JT + j] = s;
    }
  __syncthreads();
  if (t < KT * JT) {
    const float s = (float)(((double)sums[0][t] + (double)sums[1][t]) + ((double)sums[2][t] + (double)sums[3][t]));
    if (p.splits > 1) {
      p.part[(((size_t)g * p.tilesI * p.tilesJ + blockIdx.x) * p.splits + split) * (KT * JT) + t] = s;
    } else {
      const int i = it * KT + t / JT, j = jt * JT + t % JT;
      if (i < p.Kg && j < p.J) p.out[((size_t)g * p.Kg + i) * p.J + j] = s;
    }
  }
}

// dw[e] = sum of its piece's partial sums: one wave per element, lanes along the splits.
__global__ __launch_bounds__(kThreads) void narrow_sum(const float* __restrict__ part, float* __restrict__ out, int Kg, int J, int tilesI,
                                                       int tilesJ, int splits, int KT, int JT, int elements) {
  const int e = (int)blockIdx.x * (kThreads / tt::kWave) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (e >= elements) return;
  const int g = e / (Kg * J), rest = e - g * Kg * J, i = rest / J, j = rest - i * J;
  const size_t tile = (size_t)g * tilesI * tilesJ + (size_t)(j / JT) * tilesI + i / KT;
  const float* __restrict__ from = part + tile * splits * (KT * JT) + (i % KT) * JT + j % JT;
  double s = 0.0;
  for (int k = lane; k < splits; k += tt::kWave) s += (double)from[(size_t)k * (KT * JT)];
  for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, tt::kWave);
  if (lane == 0) out[e] = (float)s;
}

// ---- host side -----------------------------------------------------------------------------------------

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

template <int KT, int PX, bool BF>
void launch_conv(const NarrowConv& p, int blocks, hipStream_t st) {
  const dim3 grid(blocks, p.groups);
  if (p.epi.on) p.A < 4 ? conv_narrow<KT, PX, BF, true, true><<<grid, kThreads, 0, st>>>(p) : conv_narrow<KT, PX, BF, false, true><<<grid, kThreads, 0, st>>>(p);
  else p.A < 4 ? conv_narrow<KT, PX, BF, true, false><<<grid, kThreads, 0, st>>>(p) : conv_narrow<KT, PX, BF, false, false><<<grid, kThreads, 0, st>>>(p);
}
template <bool BF>
void launch_conv(const NarrowConv& p, int px, int blocks, hipStream_t st) {
  if (p.I <= 4) px > 1 ? launch_conv<4, 4, BF>(p, blocks, st) : launch_conv<4, 1, BF>(p, blocks, st);
  else if (p.I <= 8) px > 1 ? launch_conv<8, 4, BF>(p, blocks, st) : launch_conv<8, 1, BF>(p, blocks, st);
  else px > 1 ? launch_conv<16, 2, BF>(p, blocks, st) : launch_conv<16, 1, BF>(p, blocks, st);
}
template <int KT, int JT>
void launch_wgrad(const NarrowWgrad& p, bool bf16, hipStream_t st) {
  const dim3 grid(p.tilesI * p.tilesJ, p.groups, p.splits);
  if (bf16) wgrad_narrow<KT, JT, true><<<grid, kThreads, 0, st>>>(p);
  else wgrad_narrow<KT, JT, false><<<grid, kThreads, 0, st>>>(p);
}

int g_narrow = 1;   // tests: 0 = never, 2 = wherever they can

}  // namespace

namespace ttc {

// Measured against the matrix kernels over 250 launches of 1 to 16 rows.  A chain takes 50 to 170 ns a step here,
// by rows, and what those lose in empty rows takes many pixels to show; but they need a launch to lay out the weights,
// and another to clear dx where a stride leaves pixels without a tap.
//   short chains: 72 steps on 8 images of 28x28, 4 rows 10.3 -> 7.7 us, 8 rows 10.3 -> 8.7, 12 rows 10.3 and 16.3; 576 steps of 4
//     rows 15.3 and 34.
//   three blocks of pixels per compute unit and more: 64 images of 56x56, 576 steps of 4, 8 and 12 rows 99 -> 64, 97 -> 77, 97
//     and 129; 2304 steps of 4 and 8 rows 334 -> 235, 326 -> 279; 1024 steps at stride 2, 3 rows, 100 -> 86.
//   input gradients of a strided layer (several classes): 78 steps of 8 rows 19.1 -> 10.4, 32 of 8 15.9 -> 9.5, 26 of 12 13.3 -> 9.0,
//     200 of 8 13.4 and 20.0, 80 of 10 16.4 and 19.9; at stride 1 with fewer pixels no clear gain (30 steps of 3
//     rows on 2 of 182x182 12.2 and 12.3).
//     -- up to 6e8 products over 4, 8 or 16 rows where those stack the classes of a layer as rows of one launch: 3 rows,
//     1024 steps, 64 images of 224x224 (a 7x7 stem) 727 us and 327; 256 steps, 64 of 128x128 85, 72; 128 of 64x64 51, 58;
//     7 rows, 80 steps, 2.9e6 pixels 148, 65.  (2064 such launches: 39.5 ms here, 39.7 there, 31.9 with this line, 31.1 at best.)
//   steps that fill whole chunks of 16, whose weights those read in place: 64 steps of 2 to 8 rows 9.7 to 14.2 us and 6.6 to 6.8, 48 of up to 4 rows 7.1, 6.6.
// (bf16 arithmetic, whose matrix kernels take half the time: 45 steps of 12 rows on 147 images of 18x53 17 and 30 us, so
// more than eight rows stay with those, and long chains; of 5 to 8 rows at unit stride from 37 steps on (63 steps of 7 rows
// on 54 of 118x213 71, 46), of classes stacked as rows from 5e7 products.)
bool narrow_conv_takes(const NarrowConv& p, bool bf16) {
  if (g_narrow == 0 || p.I > 16 || p.n < 1) return false;
  long long pixels = 0, steps = 0;
  for (int i = 0; i < p.n; ++i) {
    // byte offsets relative to a block's first image
    const long long span = 1023 / ((long long)p.c[i].U * p.c[i].V) + 2;
    if (4 * ((span + 1) * p.srcN) >= (1LL << 31) - (1LL << 20)) return false;
    pixels += p.c[i].M;
    steps = std::max(steps, (long long)p.A * p.c[i].TB * p.c[i].TC);
  }
  if (g_narrow == 2) return true;
  const bool few = p.I <= 8;
  if (bf16 && !few) return false;
  // the matrix kernels take all classes of an ungrouped layer as rows of one launch
  const int rows = p.I <= 4 ? 4 : few ? 8 : 16;
  if (p.n > 1 && p.groups == 1 && p.n * p.I <= 64 && (double)pixels * rows * steps > (bf16 ? 5e7 : 6e8)) return false;
  if (p.n == 1 && bf16 && p.I > 4 && steps > 36) return false;
  if (pixels * p.groups >= 3LL * kThreads * tt::compute_units() && steps <= (!few ? 24 : bf16 ? 128 : 2560)) return true;
  if (p.n > 1) return steps <= (few ? 96 : 32);
  // (steps in whole chunks: they read the weights in place)
  return !p.gradient && steps <= (!few ? 24 : steps % 16 == 0 ? 48 : 72);
}

int narrow_conv_launch(NarrowConv& p, bool bf16, int prof_id, int* plan8) {
  tt::ProfScope prof(prof_id);
  long long pixels = 0;
  for (int i = 0; i < p.n; ++i) pixels += p.c[i].M;
  const int px_many = p.I <= 8 ? 4 : 2;
  // several pixels per thread where that leaves four blocks per compute unit
  const int px = pixels * p.groups >= 4LL * tt::compute_units() * kThreads * px_many ? px_many : 1;
  int blocks = 0;
  for (int i = 0; i < p.n; ++i) {
    p.c[i].block0 = blocks;
    p.c[i].divTaps = tt::make_fastdiv((uint32_t)std::max(1, p.c[i].TB * p.c[i].TC));
    blocks += ceil_div(p.c[i].M, kThreads * px);
  }
  p.divUnit = tt::make_fastdiv((uint32_t)(4 * p.A));
  const int rows = p.I <= 4 ? 4 : p.I <= 8 ? 8 : 16;
  const int plan[8] = {rows, kThreads * px, blocks, 1, -3, blocks, 0, 0 | (bf16 ? 1 : 0) << 8};
  std::copy(plan, plan + 8, plan8);
  bf16 ? launch_conv<true>(p, px, blocks, tt::stream()) : launch_conv<false>(p, px, blocks, tt::stream());
  TT_LAUNCH_CHECK();
  return 0;
}

bool narrow_wgrad_takes(NarrowWgrad& p, bool bf16) {
  if (g_narrow == 0 || p.R * p.S > 31) return false;
  const long long span = 255 / (long long)p.PQ + 2;
  const long long reach = 4 * ((span + 1) * std::max(p.xN, p.dyN) + 2LL * p.xBias + ((long long)p.H + p.ph + (long long)p.R * p.dh + 2) * p.W +
                               p.pw + (long long)p.S * p.dw);
  if (reach >= (1LL << 31) - (1LL << 20)) return false;
  p.KT = p.Kg <= 4 ? 4 : p.J <= 4 ? 16 : 8;
  p.JT = 64 / p.KT;
  p.tilesI = ceil_div(p.Kg, p.KT);
  p.tilesJ = ceil_div(p.J, p.JT);
  const long long tiles = (long long)p.tilesI * p.tilesJ;
  if (tiles > 65535 || tiles * p.groups * 64 > (1LL << 26)) return false;
  // about eight blocks per compute unit, each with at least four pixels per thread
  const long long want = std::max(1LL, 8LL * tt::compute_units() / (tiles * p.groups));
  p.perSplit = (int)std::max<long long>(4 * kThreads, (p.M + want - 1) / want);
  p.perSplit = ceil_div(p.perSplit, kThreads) * kThreads;
  p.splits = ceil_div(p.M, p.perSplit);
  if (p.splits > 65535) return false;
  if (g_narrow == 2) return p.Kg <= 16 || p.J <= 16;
  // 1 and 8 rows x 576 columns, 64 images of 56x56: 155 -> 53 us and 157 -> 97; 32 groups of 1 x 9: 259 -> 33.  Up to
  // sixteen rows where there are few columns (12 x 72, 64 of 56x56 51.6 -> 33.8; 9 x 1056 31 and 40).  Not few pixels:
  // those kernels add their partial sums themselves (1x1, 1 x 64, 8 of 28x28: 11.6 and 12.6; 8 x 657 of 1309 pixels 12.7
  // and 15.8).
  const bool fits = p.Kg <= 8 || p.J <= 8 || (p.Kg <= 16 && p.J <= 96);
  const bool taps = p.R * p.S > 1;
  if (!fits || (taps ? p.M < 4096 && p.J > 128 : p.M < 16384)) return false;
  // Over 6780 launches that are left (144.2 ms here, 214.6 on the matrix kernels) one in seventeen was more than 8 % slower
  // here; most of them are among these, which go back (142.8 ms, and one in a hundred):
  //   sums that take the second launch, of up to 64 columns: one tile there, added in place (1103 launches 14.2 -> 13.4 ms);
  if (taps && p.J <= 64 && p.splits > 1 && p.M < (bf16 && p.J > 16 ? 16384 : 8192)) return false;
  //   a chain or two of steps, where one block's start is all of it (166 launches 7.8 -> 7.0 us each);
  if (taps && p.M <= 128 && p.J > 8 && p.J <= 128) return false;
  //   and in bf16 arithmetic many products a fetched value: the matrix kernels take half the time (41 of more than eight
  //   rows 33 -> 29 us each, 65 of five to eight 90 -> 85).
  if (bf16 && (p.Kg > 8 ? p.J > 32 && p.M > 32768 : p.Kg > 4 && p.J > 1024)) return false;
  return true;
}
size_t narrow_wgrad_workspace(const NarrowWgrad& p) {
  return p.splits > 1 ? sizeof(float) * 64 * (size_t)p.tilesI * p.tilesJ * p.groups * p.splits : 0;
}
int narrow_wgrad_launch(NarrowWgrad& p, bool bf16) {
  void* ws = nullptr;
  if (p.splits > 1 && tt::workspace(narrow_wgrad_workspace(p), &ws)) return -1;
  p.part = (float*)ws;
  hipStream_t st = tt::stream();
  {
    tt::ProfScope prof(TT_PROF_CONV_WGRAD);
    if (p.KT == 4) launch_wgrad<4, 16>(p, bf16, st);
    else if (p.KT == 8) launch_wgrad<8, 8>(p, bf16, st);
    else launch_wgrad<16, 4>(p, bf16, st);
  }
  TT_LAUNCH_CHECK();
  if (p.splits > 1) {
    tt::ProfScope prof(TT_PROF_CONV_WGRAD_REDUCE);
    const int elements = p.groups * p.Kg * p.J;
    narrow_sum<<<ceil_div(elements, kThreads / tt::kWave), kThreads, 0, st>>>(p.part, p.out, p.Kg, p.J, p.tilesI, p.tilesJ, p.splits, p.KT,
                                                                             p.JT, elements);
    TT_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace ttc

extern "C" int tt_conv2d_narrow_enable(int on) {
  TT_API_LOCK();
  TT_REQUIRE(on >= 0 && on <= 2, "tt_conv2d_narrow_enable: %d is out of range (0..2)", on);
  g_narrow = on;
  return 0;
}
