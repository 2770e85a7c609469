// Pieces shared by the GEMM kernels that stage their operands through LDS with
// LDS-DMA loads (mb_gemm.hip, mb_gemm_ring.h).
#pragma once

#include <cstdint>
#include <type_traits>

#include "mb_gemm_offsets.h"
#include "mb_internal.h"
#include "mb_mfma.h"

namespace mb {

constexpr int kXcds = 8;

// One 16-byte-per-lane LDS DMA: lane l's 16 bytes land at the LDS address in m0
// + 16 * l. Issued as inline assembly so the compiler's wait-count pass does not
// force a full vmcnt(0) before every LDS read; the staged kernel issues it ahead
// of compiler-visible loads, whose in-order vmcnt waits then cover it.
//
// The load needs a wait state after the scalar write of m0, which the compiler
// puts for its own LDS loads only. dma16 does both, with a wait state. The
// all-DMA 256x256 kernels' loops, where that costs 1.2% (BF16 8192^3 719 -> 728
// us), write m0 (dma_address) a block update before the load (dma16_at) instead:
// 695 us where the write directly before the load takes 701.
__device__ __forceinline__ uint32_t dma_address(uint32_t lds, uint32_t lds_add) {
  uint32_t m0;
  asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(m0) : "s"(lds), "s"(lds_add) : "scc");
  return m0;
}

__device__ __forceinline__ void dma16_at(uint32_t m0, __amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voffset), "s"(rsrc), "s"(soffset), "{m0}"(m0)
               : "memory");
}

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset, uint32_t lds,
                                      uint32_t lds_add) {
  asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voffset), "s"(rsrc),
               "s"(soffset), "s"(lds), "s"(lds_add)
               : "m0", "scc", "memory");
}

// Word 3 of a gfx9 buffer resource: 32-bit data format, no swizzle, raw offsets.
constexpr int kBufferWord3 = 0x00020000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const uint8_t* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, bytes, kBufferWord3);
}

// Tile (tile_m, tile_n) of workgroup blockIdx.x: XCD-first numbering, then
// GROUP_M-row bands (see the file comment).
__device__ __forceinline__ void band_tile(int tiles_m, int tiles_n, int group_m, int& tile_m, int& tile_n) {
  const int count = gridDim.x;
  int pid = blockIdx.x;
  if (count % kXcds == 0) pid = (pid % kXcds) * (count / kXcds) + pid / kXcds;
  const int band = group_m * tiles_n;
  const int first_m = (pid / band) * group_m;
  const int rows_in_band = min(tiles_m - first_m, group_m);
  tile_m = first_m + (pid % band) % rows_in_band;
  tile_n = (pid % band) / rows_in_band;
}

// Tile of workgroup blockIdx.x for any grid size: XCD x (ids x, x+8, ..) owns
// a contiguous share of the band order, the first count % 8 XCDs one tile more.
__device__ __forceinline__ void band_tile_any(int tiles_m, int tiles_n, int group_m, int& tile_m, int& tile_n) {
  const int count = gridDim.x, xcd = blockIdx.x % kXcds, index = blockIdx.x / kXcds;
  const int pid = xcd * (count / kXcds) + min(xcd, count % kXcds) + index;
  const int band = group_m * tiles_n;
  const int first_m = (pid / band) * group_m;
  const int rows_in_band = min(tiles_m - first_m, group_m);
  tile_m = first_m + (pid % band) % rows_in_band;
  tile_n = (pid % band) / rows_in_band;
}

// s_waitcnt's immediate for vmcnt(n) alone (n < 64): vmcnt's low four bits
// at 3:0 and high two at 15:14, expcnt (6:4) and lgkmcnt (11:8) at their
// maxima, which wait for nothing.
constexpr int vmcnt_only(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// s_waitcnt's immediate for lgkmcnt(0) alone.
constexpr int kLgkmcntZero = 15 | (3 << 14) | (7 << 4);

// Barrier that orders LDS only: global loads in flight stay in flight across
// it. The LDS reads before it are waited for explicitly: at a loop's head the
// compiler drops the wait that the release fence asks for when nothing is
// outstanding on the way into the loop, though reads of the last trip are.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(kLgkmcntZero);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f(integral_constant<I>) for I = I0 .. N-1, so counts derived from I are constants.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

}  // namespace mb
