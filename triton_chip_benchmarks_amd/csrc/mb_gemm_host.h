// Host-side record of a GEMM kernel, shared by the translation units that
// instantiate them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mb {

// Launchers size their own grid: one workgroup per output tile of their kernel.
using GemmLauncher = void (*)(const uint8_t*, const uint8_t*, const uint8_t*, const uint8_t*, void*, int, int, int,
                              int, hipStream_t);

inline uint32_t tile_count(int m, int n, int bm, int bn) {
  return static_cast<uint32_t>(((m + int64_t{bm} - 1) / bm) * ((n + int64_t{bn} - 1) / bn));
}

// What one round of a kernel's workgroups (`resident` per CU on 256 CUs) takes,
// in microseconds: `tile` once (prologue, epilogue) and, per 128-byte K step,
// from `step_empty` to `step_full` with the filled share of the round. That is
// the chip's share where operand traffic and the power limit slow a step down as
// more CUs run. FP32 (`per_cu`) waits for the matrix cores of the busiest CU:
// 257 tiles of a pair take as long as 512. After full rounds the rest spreads
// less evenly, as CUs become free: halfway to a full one.
struct GemmCost {
  float tile, step_empty, step_full;
  bool per_cu;
};

struct GemmKernel {
  int format;
  int tile_m, tile_n;
  int default_group;  // band height in tile rows when the caller passes 0
  int resident;       // workgroups a CU holds at once
  GemmCost cost;
  const char* name;
  const void* kernel;
  GemmLauncher launch;
};

// BF16, FP16, FP8 and INT8, fitted to 317 launches on an MI355X (M, N from 256 to
// 8192, 2 to 64 K steps) when the ring kernels were first written. On the kernels
// as they are, over 4800 shapes (M, N from 32 to 11000, 1 to 370 steps), the
// cheapest estimate runs the fastest kernel or one within 2% of it in 88 to 93% of
// them and costs 0.7 (BF16) to 1.1% (FP8) on average; always 256x256 costs 143%.
// One launch in 73 loses over 15%, typically 2.4 us, mostly on 64x64 tiles of which
// a CU has two or three where one of 128x128 is faster; the worst are 54% (6.7 us)
// and 98 us (15%). The ragged 256x256 kernel shares kCost256: where both can
// run it takes 0.94 to 1.04 times the exact one's time.
constexpr GemmCost kCost256{7.4f, 0.85f, 1.41f, false};
constexpr GemmCost kCost256x128{4.5f, 0.44f, 0.855f, false};
constexpr GemmCost kCost128{2.9f, 0.255f, 0.48f, false};
constexpr GemmCost kCost128Pair{2.0f, 0.39f, 1.04f, false};
constexpr GemmCost kCost64{1.45f, 0.105f, 0.575f, false};
// MXFP4, whose step is four times the operations of BF16's for the same bytes,
// fitted to 530 shapes: 0.5% over the fastest on average (the constants above:
// 1.5% over 350 of them), at most 24% (14 us). Its stages carry scales, so a CU holds two of its 64x64 tiles; priced
// with three, they ran where 128x128 is faster (8704x256x3584 12.4 us, 128x128
// 9.6).
constexpr GemmCost kCostMx256{12.66f, 0.75f, 1.806f, false};
constexpr GemmCost kCostMx256x128{6.73f, 0.551f, 1.049f, false};
constexpr GemmCost kCostMx128{4.47f, 0.317f, 0.621f, false};
constexpr GemmCost kCostMx128Pair{3.63f, 0.661f, 1.247f, false};
constexpr GemmCost kCostMx64{2.04f, 0.213f, 0.555f, false};
// FP32 and FP64, fitted to 545 and 580 shapes (M, N from 128 to 16384, 2 to 512
// steps, half of them exact) on the kernels that take them: the cheapest estimate
// costs 0.17% and 0.09% on average against the fastest, at most 10% (19 us) and
// 5%, and never over 2% more than the largest tile. FP32 8192^3 7432 -> 7166 us,
// 3072x10240x7744 3607 -> 3402; FP64 512x14848x1856 444 -> 419: a dearer largest
// tile and, for FP32, the chip's share kept that tile from running.
constexpr GemmCost kCostF32x256{9.67f, 7.11f, 7.11f, true};
constexpr GemmCost kCostF32x128{4.71f, 1.974f, 1.974f, true};
constexpr GemmCost kCostF32x128Pair{4.53f, 0.404f, 3.58f, true};
constexpr GemmCost kCostF32x64{1.87f, 0.02f, 1.52f, true};
constexpr GemmCost kCostF64x256{9.5f, 3.6f, 3.7f, false};
constexpr GemmCost kCostF64x128{5.5f, 1.7f, 1.97f, false};
constexpr GemmCost kCostF64x64{1.3f, 0.2f, 1.53f, false};

// The ring kernels (mb_gemm_ring.h), compiled in mb_gemm_ring.hip.
const GemmKernel* ring_kernels(int* count);

}  // namespace mb
