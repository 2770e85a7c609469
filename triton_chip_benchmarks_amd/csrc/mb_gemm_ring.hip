// The ring GEMM kernels of every format (see mb_gemm_ring.h).
#include "mb_gemm_ring.h"

#include "mb_gemm_host.h"

namespace mb {
namespace {

template <class Op, int BM, int BN, int STAGES>
void launch_ring(const uint8_t* a, const uint8_t* b, const uint8_t* sa, const uint8_t* sb, void* c, int m, int n,
                 int k, int group_m, hipStream_t stream) {
  gemm_ring_kernel<Op, BM, BN, STAGES><<<dim3(tile_count(m, n, BM, BN)), dim3(256), 0, stream>>>(
      a, b, sa, sb, static_cast<typename Op::Out*>(c), m, n, k, group_m);
}

// BAND is the default band height, in tile rows. An XCD takes consecutive
// tiles, 32 a round where a CU holds one, and the band's shape decides which
// panels they share in its L2. Over 11 shapes of 5 formats against 8 rows:
// 128x128 takes 3.4 % less with 6 (2.7 % with 4; FP8 2048^3 11.5 -> 11.1 us,
// 6000x512x2048 10.2 -> 9.2, never over 0.5 % more), 256x128 3.7 % less with 4
// (FP8 8192x1024x2048 22.6 -> 19.4 us, BF16 35.8 -> 33.5); the pairs take 1.1 %
// more with 6 and 64x64 is level, so both keep 8. BF16 2048^3 gains 4 % (20.2 ->
// 19.4 us) with the same 12 panels an XCD and the same 50 MB of reads over the
// fabric, by counter: there it is not the bytes, and what it is stays open.
// The workgroups a CU holds are bounded by LDS: the kernels take at most 228
// (pair) and 108 (64x64) of a SIMD's 512 registers a lane.
#define MB_RING(FMT, OP, BM, BN, STAGES, BAND, COST, NAME)                                                   \
  GemmKernel {                                                                                               \
    FMT, BM, BN, BAND, RingTile<OP, BM, BN, STAGES>::RESIDENT, COST, NAME,                                   \
        reinterpret_cast<const void*>(gemm_ring_kernel<OP, BM, BN, STAGES>), launch_ring<OP, BM, BN, STAGES> \
  }
#define MB_RING_SET(FMT, OP, TYPE, BK, COST)                                                    \
  MB_RING(FMT, OP, 256, 128, 3, 4, COST##256x128, "gemm_" TYPE "_256x128x" BK),                 \
      MB_RING(FMT, OP, 128, 128, 4, 6, COST##128, "gemm_" TYPE "_128x128x" BK),                 \
      MB_RING(FMT, OP, 128, 128, 2, 8, COST##128Pair, "gemm_" TYPE "_128x128x" BK "_pair"),     \
      MB_RING(FMT, OP, 64, 64, 3, 8, COST##64, "gemm_" TYPE "_64x64x" BK)

const GemmKernel kRingKernels[] = {
    MB_RING_SET(MB_MATRIX_BF16, MfmaBf16, "bf16", "64", kCost),
    MB_RING_SET(MB_MATRIX_F16, MfmaF16, "f16", "64", kCost),
    MB_RING_SET(MB_MATRIX_FP8_E4M3, MfmaFp8, "fp8", "128", kCost),
    MB_RING_SET(MB_MATRIX_I8, MfmaI8, "i8", "128", kCost),
    MB_RING_SET(MB_MATRIX_MXFP4, MfmaMxfp4, "mxfp4", "256", kCostMx),
    // FP32 and FP64 are bound by the matrix cores at every tile: no 256x128.
    MB_RING(MB_MATRIX_F32, MfmaF32, 128, 128, 4, 6, kCostF32x128, "gemm_f32_128x128x32"),
    MB_RING(MB_MATRIX_F32, MfmaF32, 128, 128, 2, 8, kCostF32x128Pair, "gemm_f32_128x128x32_pair"),
    MB_RING(MB_MATRIX_F32, MfmaF32, 64, 64, 3, 8, kCostF32x64, "gemm_f32_64x64x32"),
    MB_RING(MB_MATRIX_F64, MfmaF64, 128, 128, 4, 6, kCostF64x128, "gemm_f64_128x128x16"),
    MB_RING(MB_MATRIX_F64, MfmaF64, 64, 64, 3, 8, kCostF64x64, "gemm_f64_64x64x16"),
};

struct RingRegistrar {
  RingRegistrar() {
    for (const GemmKernel& kernel : kRingKernels) register_kernel(kernel.name, kernel.kernel);
  }
};
const RingRegistrar kRingRegistrar;

}  // namespace

const GemmKernel* ring_kernels(int* count) {
  *count = static_cast<int>(sizeof(kRingKernels) / sizeof(kRingKernels[0]));
  return kRingKernels;
}

}  // namespace mb
