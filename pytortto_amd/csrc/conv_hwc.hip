// Convolutions with operands rounded to bfloat16 (TT_CONV_MATH_BF16), channel-last: the kernels behind
// Conv2d forward and the stride-1 input gradient where the reduction is long.
//
//   D[i, m] = sum over taps t and channels c of  W[i][t][c] * X[pixel(m, t)][c]      (+ epilogue)
//
// The other kernels gather x in place, one 4-byte element per lane and tap, and round it behind that: a
// 3x3 layer fetches and converts every element nine times, and the address unit, not the matrix pipe,
// sets its speed.  Here a first pass over x rounds every element once and lays the channels of a pixel
// out contiguously; the product then fetches 16 bytes (eight channels) per lane, for any tap, and writes
// them to LDS as they are.  The pass costs one read of x and one write of its 2 bytes per element; the
// layouts live in the library's workspace for the length of a call.
// Measured, batch 64, forward, random operands, 14.8 GFLOP each; the whole call in the other kernels, here, and
// of that the product: 512 channels 7x7 80.5 us, 49.1, 27.9 (530 TFLOP/s); 256 channels 14x14 72.9, 49.1,
// 30.6 (484), the same at stride 2 80.6, 57.0, 30.2; 128 channels 28x28 43.8, 42.5, 30.4; 64 channels 56x56
// 50.2, 63.6, 44.9 (330): the rule in hwc_supported.
// No unit bounds the product: the matrix pipe and the LDS are each busy for a fifth of its cycles (0.17 to
// 0.19, no bank conflicts).  It is a chain of fetch, LDS and matrix instructions per chunk, with a barrier, in two
// blocks per compute unit.
// (In three bfloat16 terms per element the same kernels were no faster than the gathering ones: six
// products read three times the bytes, and 6 bytes per element are written and read around them.)
//
// One chunk of the reduction is a tap and 64 channels of it: 128 bytes of a row or pixel, contiguous; in
// LDS at a pitch of 144, which spreads any eight consecutive rows over all banks for the 16-byte accesses.
#include <algorithm>
#include <cstdlib>

#include "conv_igemm_common.h"

namespace {

using namespace ttc;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 64;              // channels of a chunk
constexpr int kOct = kBK / 8;        // 16-byte units of its rows
constexpr int kBytes = 16 * kOct;
constexpr int kPitch = kBytes + 16;  // in LDS

__device__ __forceinline__ unsigned pack2(float lo, float hi) {
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(unsigned, v);
}

__device__ __forceinline__ uintx4 round8(const float (&v)[8]) {
  return uintx4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
}

// ---- x[n][c][h][w] -> xt[pixel of the batch][c] in bfloat16, channels padded with zeros to whole chunks -----
// A block takes 64 pixels x 64 channels: reads coalesced along the pixels, all sixteen loads of a thread in
// flight together, writes the 128 bytes of a pixel next to each other, through LDS.  Bound by memory.
__global__ __launch_bounds__(kThreads) void channels_last(const float* __restrict__ x, uintx4* __restrict__ xt, int C, int Cp,
                                                         uint32_t pixels, tt::FastDiv divHW) {
  constexpr int kLine = kOct + 1;
  __shared__ uintx4 tile[64 * kLine];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t p0 = blockIdx.x * 64, px = min(p0 + lane, pixels - 1);
  const int c0 = blockIdx.y * kBK;
  const uint32_t n = tt::fd_div(px, divHW);
  const size_t HW = divHW.d;
  const float* __restrict__ src = x + (size_t)n * C * HW + (px - n * divHW.d);
  float v[2][8];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int c = c0 + 8 * (wave * 2 + j) + e;       // wave-uniform
      v[j][e] = c < C ? src[(size_t)c * HW] : 0.f;
    }
#pragma unroll
  for (int j = 0; j < 2; ++j) tile[lane * kLine + wave * 2 + j] = round8(v[j]);
  __syncthreads();
  const size_t pitch = (size_t)Cp / 8;
  uintx4* __restrict__ dst = xt + (size_t)p0 * pitch + c0 / 8;
#pragma unroll
  for (int u = threadIdx.x; u < 64 * kOct; u += kThreads) {
    const int row = u / kOct, k = u % kOct;
    if (p0 + row < pixels) dst[row * pitch + k] = tile[row * kLine + k];
  }
}

// ---- weights -> wt[row][tap][c], rows and channels padded with zeros -----------------------------------
// forward: row k, w[k][c][tap];  input gradient: row c, channel k, taps in reverse order.  One thread per
// row, tap and eight channels.
template <bool DGRAD>
__global__ __launch_bounds__(kThreads) void pack_weights(const float* __restrict__ w, uintx4* __restrict__ wt, int rows, int chans,
                                                        int taps, int Cp, int total) {
  const int u = blockIdx.x * kThreads + threadIdx.x;
  if (u >= total) return;
  // forward: taps innermost (contiguous in w); input gradient: rows innermost but for the taps
  const int octs = Cp / 8;
  const int rest = u / taps, tap = u - rest * taps;
  int row, o;
  if constexpr (DGRAD) {
    const int padded = total / (taps * octs);
    o = rest / padded;
    row = rest - o * padded;
  } else {
    row = rest / octs;
    o = rest - row * octs;
  }
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = 8 * o + e;
    const bool ok = row < rows && c < chans;
    v[e] = !ok ? 0.f
               : DGRAD ? w[((size_t)c * rows + row) * taps + (taps - 1 - tap)] : w[((size_t)row * chans + c) * taps + tap];
  }
  wt[((size_t)row * taps + tap) * octs + o] = round8(v);
}

// ---- the product -------------------------------------------------------------------------------------
struct Hwc {
  const char* xt;
  const char* wt;
  float* partial;      // splits > 1: [splits][elements of out] sums over a part of the chunks each
  long long outElems;
  int cchunks;         // chunks of one tap
  int chunks;          // taps * cchunks
  int perSplit;
  int S;               // tap t = (t / S, t % S)
  int rowBytes;        // of wt
  int pixBytes, imgBytes;   // of xt
  int bias;            // bytes added to every pixel offset so that it is never negative
  int tapRow, tapCol;  // byte steps of a tap row / column
  int stepH, stepW;    // the same in pixels, for the bounds
  int R;
};

// Tile 64*MT rows x 64*NT pixels, four waves as 2 x 2, MT x NT accumulators of 32 x 32 each.  Every thread
// fetches the same 16-byte units of the chunk each time (their rows, pixels and taps outside the image are
// fixed for the tile), one chunk ahead of the matrix instructions; two LDS buffers, one barrier per chunk.
template <int MT, int NT>
__global__ __launch_bounds__(kThreads, 2) void hwc_product(const Igemm p, const Hwc q) {
  constexpr int BM = 64 * MT, BN = 64 * NT, kRows = BM + BN;
  constexpr int kAUnits = BM * kOct, kUnits = kRows * kOct;
  constexpr int IT = kUnits / kThreads;
  static_assert(kAUnits % kThreads == 0 && kUnits % kThreads == 0, "an item is a unit of the weights or of the pixels for all threads");
  __shared__ __align__(16) char lds[2][kRows * kPitch];
  __shared__ __align__(16) float epi_lds[4 * BM];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int tile = tt::xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int tilesI = p.Ipad / BM;
  const int i0 = (tile % tilesI) * BM;
  const int m0 = (tile / tilesI) * BN;
  const int q0 = (int)blockIdx.z * q.perSplit, q1 = min(q.chunks, q0 + q.perSplit);

  const uint32_t n0 = tt::fd_div((uint32_t)__builtin_amdgcn_readfirstlane(m0), p.divUV);   // first image of the tile
  const __amdgpu_buffer_rsrc_t xSrd =
      __builtin_amdgcn_make_buffer_rsrc((void*)(q.xt + (long long)n0 * q.imgBytes - q.bias), 0, kSrdRecords, kSrdFlags);
  const __amdgpu_buffer_rsrc_t wSrd = __builtin_amdgcn_make_buffer_rsrc((void*)q.wt, 0, kSrdRecords, kSrdFlags);

  int voff[IT], at[IT];
  uint32_t outside[IT];   // bit t set: tap t lies outside the image for this unit's pixel
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int u = it * kThreads + tid;
    const int row = u / kOct, oct = u - row * kOct;
    at[it] = row * kPitch + 16 * oct;
    outside[it] = 0;
    if (it * kThreads < kAUnits) {
      voff[it] = (i0 + row) * q.rowBytes + 16 * oct;
    } else {
      voff[it] = 16 * oct;
      outside[it] = ~0u;
      const int m = m0 + row - BM;
      if (m < p.M) {
        const uint32_t n = tt::fd_div((uint32_t)m, p.divUV);
        const uint32_t rem = (uint32_t)m - n * p.divUV.d;
        const uint32_t pu = tt::fd_div(rem, p.divV);
        const uint32_t pv = rem - pu * p.divV.d;
        const int ih = (int)pu * p.su + p.bh, iw = (int)pv * p.sv + p.bw;
        voff[it] += (int)(n - n0) * q.imgBytes + (ih * p.Wlim + iw) * q.pixBytes + q.bias;
        uint32_t cols = 0, inside = 0;
        for (int c = 0; c < q.S; ++c) cols |= (uint32_t)((unsigned)(iw + c * q.stepW) < (unsigned)p.Wlim) << c;
        for (int r = 0; r < q.R; ++r)
          if ((unsigned)(ih + r * q.stepH) < (unsigned)p.Hlim) inside |= cols << (r * q.S);
        outside[it] = ~inside;
      }
    }
  }

  // position of the chunk being fetched
  int fq = q0, ftap = q0 / q.cchunks, fc = q0 - ftap * q.cchunks, fr = ftap / q.S, fs = ftap - fr * q.S;
  uintx4 reg[IT];
  auto fetch = [&]() __attribute__((always_inline)) {
    const int woff = fq * kBytes, xoff = fr * q.tapRow + fs * q.tapCol + fc * kBytes;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      if (it * kThreads < kAUnits) {
        reg[it] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(wSrd, voff[it], woff, 0));
      } else {
        const uint32_t vo = ((outside[it] >> ftap) << 31) | (uint32_t)voff[it];
        reg[it] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(xSrd, (int)vo, xoff, 0));
      }
    }
    ++fq;
    if (++fc == q.cchunks) {
      fc = 0;
      ++ftap;
      if (++fs == q.S) {
        fs = 0;
        ++fr;
      }
    }
  };
  auto stage = [&](const int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      *reinterpret_cast<uintx4*>(&lds[buf][at[it]]) = reg[it];
    }
  };

  floatx16 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  // A lane's operand of a matrix step: channels 8h .. 8h + 7 of the step, one 16-byte unit.
  const int arow = (wm * MT * 32 + l32) * kPitch + 16 * h;
  const int brow = (BM + wn * NT * 32 + l32) * kPitch + 16 * h;
  // The chunk is summed on its own, then added: 4 products in a chain and one addition per chunk, where a
  // single chain over all chunks loses more to its roundings than the kernels that gather in place do,
  // whose blocks share a reduction (against float64 sums of the rounded operands, 128 channels 28x28,
  // 3x3, batch 8: 1.35e-7 in one chain, 8.4e-8 there, 7.8e-8 so; 372 channels 50x9: 2.4e-7, 1.3e-7, 1.1e-7).
  // The additions cost 2 % of 24 calls of ResNet-50's layers at batch 8, 32 and 64 (889 us, 907 with them).
  auto multiply = [&](const int buf) __attribute__((always_inline)) {
    floatx16 sum[MT][NT];
#pragma unroll
    for (int s = 0; s < kBK / 16; ++s) {
      bf16x8 a[MT], b[NT];
#pragma unroll
      for (int x = 0; x < MT; ++x) a[x] = *reinterpret_cast<const bf16x8*>(&lds[buf][arow + x * 32 * kPitch + 32 * s]);
#pragma unroll
      for (int y = 0; y < NT; ++y) b[y] = *reinterpret_cast<const bf16x8*>(&lds[buf][brow + y * 32 * kPitch + 32 * s]);
#pragma unroll
      for (int x = 0; x < MT; ++x)
#pragma unroll
        for (int y = 0; y < NT; ++y)
          sum[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x], b[y], s == 0 ? floatx16{} : sum[x][y], 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < MT; ++x)
#pragma unroll
      for (int y = 0; y < NT; ++y) acc[x][y] += sum[x][y];
  };

  const bool whole = q.partial == nullptr;
  if (whole && p.epi.on) epilogue_constants<BM>(p, 0, i0, tid, epi_lds);   // published by the barrier below
  fetch();
  stage(0);
  __syncthreads();
  for (int c = q0; c < q1; ++c) {
    const int buf = (c - q0) & 1;
    if (c + 1 < q1) fetch();              // in flight across this chunk's matrix instructions
    multiply(buf);
    if (c + 1 < q1) stage(buf ^ 1);       // the other buffer was last read before the previous barrier
    __syncthreads();
  }

  // accumulator register r of a 32x32 tile holds row 8*(r/4) + 4*h + r%4, column l32
  uint32_t obase[NT];
  bool mok[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    const int m = m0 + (wn * NT + y) * 32 + l32;
    mok[y] = m < p.M;
    const uint32_t mm = mok[y] ? (uint32_t)m : 0u;
    const uint32_t n = tt::fd_div(mm, p.divUV);
    obase[y] = (uint32_t)((int)n * p.outStrideN + (int)(mm - n * p.divUV.d));
  }
  if (whole && p.epi.on) {
    store_through_epilogue<BM, MT, NT>(p, acc, obase, mok, i0, wm * MT * 32, h, epi_lds);
    return;
  }
  float* __restrict__ out = whole ? p.out : q.partial + (size_t)blockIdx.z * (size_t)q.outElems;
  const bool biased = whole && p.bias != nullptr;
  const uint32_t hoff = (uint32_t)(4 * h * p.outStrideI);
#pragma unroll
  for (int x = 0; x < MT; ++x) {
    const int srow = __builtin_amdgcn_readfirstlane(i0 + (wm * MT + x) * 32);
    float bz[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bz[r] = biased ? p.bias[min(srow + 8 * (r >> 2) + 4 * h + (r & 3), p.I - 1)] : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // every load done before the first store: they share one counter
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = srow + 8 * (r >> 2) + (r & 3);
      float* __restrict__ rowp = out + (size_t)row * (size_t)p.outStrideI;
      if (row + 4 * h < p.I) {
#pragma unroll
        for (int y = 0; y < NT; ++y)
          if (mok[y]) rowp[obase[y] + hoff] = biased ? acc[x][y][r] + bz[r] : acc[x][y][r];
      }
    }
  }
}

// The partial sums of a split reduction added in order, and the launch's epilogue.
__global__ __launch_bounds__(kThreads) void hwc_finish(const Igemm p, const float* __restrict__ partial, int splits,
                                                      uint32_t total, tt::FastDiv divPix, tt::FastDiv divI) {
  const uint32_t stride = gridDim.x * kThreads;
  for (uint32_t e = blockIdx.x * kThreads + threadIdx.x; e < total; e += stride) {
    float v = partial[e];
    for (int s = 1; s < splits; ++s) v += partial[(size_t)s * total + e];
    const uint32_t row = tt::fd_div(e, divPix);
    const int i = (int)(row - tt::fd_div(row, divI) * divI.d);
    if (p.bias) v += p.bias[i];
    if (p.epi.on) {
      if (p.epi.norm) {
        const float sd = __fsqrt_rn(__fadd_rn(p.epi.var[i], p.epi.eps));
        v = fmaf(v - p.epi.mean[i], __fdiv_rn(p.epi.gamma ? p.epi.gamma[i] : 1.0f, sd), p.epi.beta ? p.epi.beta[i] : 0.0f);
      }
      if (p.epi.res) v += p.epi.res[e];
      if (p.epi.relu) v = (v > 0.f || v != v) ? v : 0.f;
      if (p.epi.mask) v *= p.epi.mask[e] > 0.f ? 1.f : 0.f;
    }
    p.out[e] = v;
  }
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
size_t align_up(size_t v) { return (v + 255) / 256 * 256; }

struct Plan {
  int Cp, Ipad, mt, nt, splits, perSplit, chunks;
  size_t xt, wt, partial;   // bytes of workspace
};

Plan make_plan(const HwcConv& c) {
  const int taps = c.R * c.S;
  const long long M = (long long)c.N * c.P * c.Q;
  Plan pl{};
  pl.Cp = ceil_div(c.C, kBK) * kBK;
  pl.mt = ceil_div(c.I, 128) * 2 <= ceil_div(c.I, 64) ? 2 : 1;   // the taller tile unless it pads more rows
  pl.nt = 2;
  pl.Ipad = ceil_div(c.I, 64 * pl.mt) * 64 * pl.mt;
  pl.chunks = taps * (pl.Cp / kBK);
  const long long tiles = (long long)(pl.Ipad / (64 * pl.mt)) * ceil_div(M, 64 * pl.nt);
  // a split reduction where the tiles do not give every compute unit its two blocks: an added round trip
  // of the output through memory per split, so no share below eight chunks
  const long long slots = 2LL * tt::compute_units();
  long long s = tiles * 4 <= slots * 3 ? slots / tiles : 1;
  s = s < 1 ? 1 : s > 8 ? 8 : s;
  while (s > 1 && pl.chunks / s < 8) --s;
  pl.perSplit = ceil_div(pl.chunks, s);
  pl.splits = ceil_div(pl.chunks, pl.perSplit);
  pl.xt = align_up((size_t)c.N * c.H * c.W * pl.Cp * 2);
  pl.wt = align_up((size_t)pl.Ipad * taps * pl.Cp * 2);
  pl.partial = pl.splits > 1 ? align_up(sizeof(float) * (size_t)pl.splits * c.I * M) : 0;
  return pl;
}

}  // namespace

namespace ttc {

size_t hwc_workspace(const HwcConv& c) {
  const Plan pl = make_plan(c);
  return pl.xt + pl.wt + pl.partial;
}

bool hwc_supported(const HwcConv& c, bool always) {
  const int taps = c.R * c.S;
  if (taps > 31) return false;                                             // the masks are 32 bits
  // plain matrix products read both operands as they lie; strided 1x1 layers would lay out what they skip
  const bool pointwise = taps == 1;
  if (pointwise && (c.sh != 1 || c.sw != 1 || c.ph != 0 || c.pw != 0 || (c.P * c.Q) % 4 == 0)) return false;
  const Plan pl = make_plan(c);
  if (pl.Cp / kBK > 65535) return false;                                   // the grid of channels_last
  // 32-bit offsets inside a tile's images, the weights and the whole batch's pixels
  const long long pix = 2LL * pl.Cp, img = pix * c.H * c.W;
  const long long images = 127 / ((long long)c.P * c.Q) + 2;
  const long long bias = pix * ((long long)std::abs(c.ph) * c.W + std::abs(c.pw));
  const long long reach = pix * ((long long)(c.R - 1) * c.dh * c.W + (long long)(c.S - 1) * c.dw);
  if (images * img + 2 * bias + reach >= (1LL << 31)) return false;
  if ((long long)pl.wt >= (1LL << 31) || !tt::fits_i32((long long)c.N * c.H * c.W + 64)) return false;
  if (always) return true;
  if (pl.xt + pl.wt + pl.partial > ((size_t)1 << 30)) return false;        // workspace stays with the library
  // padded channels and rows are multiplied like the others
  if (c.C < 32 || c.I < 32) return false;
  const double padding = (double)pl.Cp * pl.Ipad / ((double)c.C * c.I);
  if (padding > 1.5) return false;
  if (2.0 * c.I * c.C * taps * c.N * c.P * c.Q < 1e9) return false;        // the passes around the product cost more than it saves
  // Against the kernels that gather in place (bf16_first_supported, launch_igemm): where those run one
  // tile per block, they lose from 128 channels on (1.0-1.5 times, 3x3 to 5x5) and win below (64 channels
  // 0.7-0.9 times); where they would share few tiles' long reductions between blocks, or the reduction is no
  // whole number of their chunks, they lose (1.1-1.9 times) -- but for the 1x1 input gradient, whose
  // weights they read in place (0.9-1.1 at batch 32 and 64).
  const long long kred = (long long)c.C * taps;
  const long long tiles = (long long)ceil_div(c.I, c.I <= 64 ? 64 : 128) * ceil_div((long long)c.N * c.P * c.Q, 128);
  const bool gathers_well = kred % 32 == 0 && (tiles >= tt::compute_units() || kred <= 1024);
  if (pointwise) return !c.dgrad && !gathers_well;
  return !gathers_well || (c.C >= 128 && padding < 1.1);
}

int hwc_conv(const HwcConv& c, const float* x, const float* w, const float* bias, float* out, const Epilogue* epi, int prof_id,
             int* plan8) {
  const int taps = c.R * c.S;
  const Plan pl = make_plan(c);
  void* ws = nullptr;
  if (tt::workspace(pl.xt + pl.wt + pl.partial, &ws)) return -1;
  char* xt = (char*)ws;
  char* wt = xt + pl.xt;
  hipStream_t st = tt::stream();
  Igemm p{};
  p.bias = bias; p.out = out;
  if (epi) p.epi = *epi;
  p.I = c.I; p.Ipad = pl.Ipad; p.M = c.N * c.P * c.Q;
  p.divUV = tt::make_fastdiv((uint32_t)(c.P * c.Q));
  p.divV = tt::make_fastdiv((uint32_t)c.Q);
  p.su = c.sh; p.bh = -c.ph; p.sv = c.sw; p.bw = -c.pw;
  p.Hlim = c.H; p.Wlim = c.W;
  p.outStrideN = c.I * c.P * c.Q; p.outStrideI = c.P * c.Q;
  Hwc q{};
  q.xt = xt; q.wt = wt;
  q.partial = pl.splits > 1 ? (float*)(wt + pl.wt) : nullptr;
  q.outElems = (long long)p.I * p.M;
  q.pixBytes = 2 * pl.Cp;
  q.imgBytes = q.pixBytes * c.H * c.W;
  q.rowBytes = q.pixBytes * taps;
  q.cchunks = pl.chunks / taps; q.chunks = pl.chunks; q.perSplit = pl.perSplit;
  q.R = c.R; q.S = c.S;
  q.bias = q.pixBytes * (std::max(c.ph, 0) * c.W + std::max(c.pw, 0));
  q.tapRow = q.pixBytes * c.dh * c.W; q.tapCol = q.pixBytes * c.dw;
  q.stepH = c.dh; q.stepW = c.dw;
  {
    tt::ProfScope prof(TT_PROF_CONV_PREP);
    const uint32_t pixels = (uint32_t)(c.N * c.H * c.W);
    channels_last<<<dim3(ceil_div(pixels, 64), pl.Cp / kBK), kThreads, 0, st>>>(x, (uintx4*)xt, c.C, pl.Cp, pixels,
                                                                               tt::make_fastdiv((uint32_t)(c.H * c.W)));
    TT_LAUNCH_CHECK();
    const int total = pl.Ipad * taps * (pl.Cp / 8);
    if (c.dgrad) pack_weights<true><<<ceil_div(total, kThreads), kThreads, 0, st>>>(w, (uintx4*)wt, c.I, c.C, taps, pl.Cp, total);
    else pack_weights<false><<<ceil_div(total, kThreads), kThreads, 0, st>>>(w, (uintx4*)wt, c.I, c.C, taps, pl.Cp, total);
    TT_LAUNCH_CHECK();
  }
  const int tiles = (pl.Ipad / (64 * pl.mt)) * ceil_div(p.M, 64 * pl.nt);
  const int plan[8] = {64 * pl.mt, 64 * pl.nt, tiles, pl.Ipad / (64 * pl.mt), -2, tiles, 0, kModeTapMask | 1 << 8};
  std::copy(plan, plan + 8, plan8);
  tt::ProfScope prof(prof_id);
  const dim3 grid((unsigned)tiles, 1, (unsigned)pl.splits);
  if (pl.mt == 2) hwc_product<2, 2><<<grid, kThreads, 0, st>>>(p, q);
  else hwc_product<1, 2><<<grid, kThreads, 0, st>>>(p, q);
  TT_LAUNCH_CHECK();
  return pl.splits > 1 ? add_partials(p, q.partial, pl.splits) : 0;
}

int add_partials(const Igemm& p, const float* partial, int splits) {
  const uint32_t total = (uint32_t)p.I * (uint32_t)p.M;
  const int blocks = std::min(ceil_div(total, kThreads), 8 * tt::compute_units());
  hwc_finish<<<blocks, kThreads, 0, tt::stream()>>>(p, partial, splits, total, p.divUV, tt::make_fastdiv((uint32_t)p.I));
  TT_LAUNCH_CHECK();
  return 0;
}

}  // namespace ttc
