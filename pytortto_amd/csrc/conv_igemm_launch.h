// The kernels of conv_igemm_kernel.h in one arithmetic, and their launches: included once by a translation
// unit that defines
//   TT_IGEMM_KERNEL, TT_IGEMM_KERNEL_MULTI   the kernels' names (the second without an epilogue only)
//   TT_IGEMM_TERMS    0: float32 matrix instructions; 1: operands rounded to bfloat16; 3: three bf16 terms
//   TT_IGEMM_BLOCKS   resident blocks per compute unit to compile for
//   TT_IGEMM_EPI      whether the launches apply an epilogue (Igemm::epi)
//   TT_IGEMM_UNIT     the name the unit is known by (conv_igemm_common.h)
// One unit each: they compile in parallel.  The launch planning stays in conv_igemm.hip, which
// calls in here with the tile shape it chose.
#pragma once
#include "conv_igemm_kernel.h"

namespace {

using namespace ttc;

template <int WM, int WN, int MT, int NT, bool SK, int MODE, bool AT>
__global__ __launch_bounds__(kThreads, TT_IGEMM_BLOCKS) void TT_IGEMM_KERNEL(const Igemm p) {
  igemm_body<WM, WN, MT, NT, SK, MODE, AT, TT_IGEMM_TERMS, TT_IGEMM_EPI>(p, (int)blockIdx.x);
}

#if !TT_IGEMM_EPI
template <int WM, int WN, int MT, int NT, int MODE>
__global__ __launch_bounds__(kThreads, TT_IGEMM_BLOCKS) void TT_IGEMM_KERNEL_MULTI(const IgemmMulti m) {
  int ci = 0;
  while (ci + 1 < m.n && (int)blockIdx.x >= m.first[ci + 1]) ++ci;
  igemm_body<WM, WN, MT, NT, false, MODE, false, TT_IGEMM_TERMS, false>(m.c[ci], (int)blockIdx.x - m.first[ci]);
}
#endif

// The stream-K wait is safe only while every block of the persistent grid is resident at once.  What the
// device can hold of one instantiation is asked once (registers and LDS of the compiled kernel decide
// it); an instantiation that cannot hold that many is launched data-parallel instead, one tile per
// block: a register-count regression then costs speed, never a stalled launch.
template <int WM, int WN, int MT, int NT, int MODE, bool AT>
int resident_blocks_per_cu() {
  static int cached = -1;
  if (cached < 0) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, TT_IGEMM_KERNEL<WM, WN, MT, NT, true, MODE, AT>, kThreads, 0) != hipSuccess) {
      (void)hipGetLastError();
      n = 0;
    }
    cached = n;
  }
  return cached;
}

// Returns whether the persistent (stream-K) grid was launched.
template <int WM, int WN, int MT, int NT, int MODE, bool AT>
bool launch_mode(const Igemm& p, int groups, int sk_blocks, int forced_occupancy, hipStream_t st) {
  if (sk_blocks > 0) {
    const int held = forced_occupancy >= 0 ? forced_occupancy : resident_blocks_per_cu<WM, WN, MT, NT, MODE, AT>();
    if ((long long)held * tt::compute_units() < sk_blocks) sk_blocks = 0;   // the data-parallel launch ignores the stream-K fields
  }
  if (sk_blocks > 0) TT_IGEMM_KERNEL<WM, WN, MT, NT, true, MODE, AT><<<dim3(sk_blocks, 1), kThreads, 0, st>>>(p);
  else TT_IGEMM_KERNEL<WM, WN, MT, NT, false, MODE, AT><<<dim3(p.tiles, groups), kThreads, 0, st>>>(p);
  return sk_blocks > 0;
}

template <int WM, int WN, int MT, int NT>
bool launch_config(const Igemm& p, int groups, int sk_blocks, int forced, hipStream_t st) {
  const bool at = p.wTransStride > 0;
  if (p.mode == kModeGemm && at) return launch_mode<WM, WN, MT, NT, kModeGemm, true>(p, groups, sk_blocks, forced, st);
  if (p.mode == kModeGemm) return launch_mode<WM, WN, MT, NT, kModeGemm, false>(p, groups, sk_blocks, forced, st);
  if (p.mode == kModeTapMask && at) return launch_mode<WM, WN, MT, NT, kModeTapMask, true>(p, groups, sk_blocks, forced, st);
  if (p.mode == kModeTapMask) return launch_mode<WM, WN, MT, NT, kModeTapMask, false>(p, groups, sk_blocks, forced, st);
  if (p.mode == kModeTapMask64) return launch_mode<WM, WN, MT, NT, kModeTapMask64, false>(p, groups, sk_blocks, forced, st);
  return launch_mode<WM, WN, MT, NT, kModeCompare, false>(p, groups, sk_blocks, forced, st);
}

// smallest number of resident blocks per CU over every stream-K instantiation of one tile shape
template <int WM, int WN, int MT, int NT>
int min_resident() {
  const int all[] = {resident_blocks_per_cu<WM, WN, MT, NT, kModeGemm, true>(),    resident_blocks_per_cu<WM, WN, MT, NT, kModeGemm, false>(),
                     resident_blocks_per_cu<WM, WN, MT, NT, kModeTapMask, true>(), resident_blocks_per_cu<WM, WN, MT, NT, kModeTapMask, false>(),
                     resident_blocks_per_cu<WM, WN, MT, NT, kModeTapMask64, false>(), resident_blocks_per_cu<WM, WN, MT, NT, kModeCompare, false>()};
  int lo = all[0];
  for (int v : all) lo = v < lo ? v : lo;
  return lo;
}

#if !TT_IGEMM_EPI
template <int WM, int WN, int MT, int NT>
void launch_multi_config(const IgemmMulti& m, int groups, hipStream_t st) {
  const dim3 grid(m.first[m.n], groups);
  if (m.c[0].mode == kModeTapMask) TT_IGEMM_KERNEL_MULTI<WM, WN, MT, NT, kModeTapMask><<<grid, kThreads, 0, st>>>(m);
  else TT_IGEMM_KERNEL_MULTI<WM, WN, MT, NT, kModeCompare><<<grid, kThreads, 0, st>>>(m);
}
#endif

bool launch(const Igemm& p, int groups, int sk_blocks, int bm, int bn, int forced_occupancy, hipStream_t st) {
  if (bm == 128 && bn == 128) return launch_config<2, 2, 2, 2>(p, groups, sk_blocks, forced_occupancy, st);
  if (bm == 64 && bn == 256) return launch_config<1, 4, 2, 2>(p, groups, sk_blocks, forced_occupancy, st);
  if (bm == 32 && bn == 256) return launch_config<1, 4, 1, 2>(p, groups, sk_blocks, forced_occupancy, st);
  return launch_config<2, 2, 1, 1>(p, groups, sk_blocks, forced_occupancy, st);
}

#if TT_IGEMM_EPI
constexpr auto launch_multi = nullptr;   // the classes of a strided input gradient: no epilogue
#else
// Data-parallel launches of one tile shape and addressing mode (no stream-K, no transposed weights) as
// one grid.
void launch_multi(const IgemmMulti& m, int groups, int bm, int bn, hipStream_t st) {
  if (bm == 128 && bn == 128) launch_multi_config<2, 2, 2, 2>(m, groups, st);
  else if (bm == 64 && bn == 256) launch_multi_config<1, 4, 2, 2>(m, groups, st);
  else if (bm == 32 && bn == 256) launch_multi_config<1, 4, 1, 2>(m, groups, st);
  else launch_multi_config<2, 2, 1, 1>(m, groups, st);
}
#endif

int min_resident_blocks() {
  const int all[] = {min_resident<2, 2, 2, 2>(), min_resident<1, 4, 2, 2>(), min_resident<1, 4, 1, 2>(), min_resident<2, 2, 1, 1>()};
  int lo = all[0];
  for (int v : all) lo = v < lo ? v : lo;
  return lo;
}

}  // namespace

namespace ttc {
const IgemmUnit& TT_IGEMM_UNIT() {
  static const IgemmUnit unit = {launch, launch_multi, min_resident_blocks};
  return unit;
}
}  // namespace ttc
