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
// from `step_empty` to `step_full` with the filled share of the round - operand
// traffic and the power limit slow a step down as more CUs run.
struct GemmCost {
  float tile, step_empty, step_full;
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

// Fitted to 317 launches on an MI355X (M, N from 256 to 8192, 2 to 64 K steps;
// BF16, FP8 and MXFP4, which move the same bytes per step and matrix cycle,
// together). Picking the cheapest estimate costs 0.7% on average against
// always picking the fastest kernel; always taking the largest tile costs 126%.
constexpr GemmCost kCost256{7.4f, 0.85f, 1.41f};
constexpr GemmCost kCost256x128{4.5f, 0.44f, 0.855f};
constexpr GemmCost kCost128{2.9f, 0.255f, 0.48f};
constexpr GemmCost kCost128Pair{2.0f, 0.39f, 1.04f};
constexpr GemmCost kCost64{1.45f, 0.105f, 0.575f};
constexpr GemmCost kCostF32x256{6.7f, 6.8f, 7.4f};
constexpr GemmCost kCostF32x128{3.0f, 1.85f, 1.97f};
constexpr GemmCost kCostF32x128Pair{2.3f, 1.7f, 3.5f};
constexpr GemmCost kCostF32x64{1.5f, 0.44f, 1.55f};
constexpr GemmCost kCostF64x256{7.5f, 3.3f, 3.83f};
constexpr GemmCost kCostF64x128{4.5f, 1.78f, 1.97f};
constexpr GemmCost kCostF64x64{1.95f, 0.365f, 1.48f};

// The ring kernels (mb_gemm_ring.h), compiled in mb_gemm_ring.hip.
const GemmKernel* ring_kernels(int* count);

}  // namespace mb
