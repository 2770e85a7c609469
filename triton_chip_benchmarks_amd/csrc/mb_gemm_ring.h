// Ring GEMM kernel: 64x64, 128x128 and 256x128 tiles, any M and N, any K of
// whole 16-byte chunks per row.
#pragma once

#include "mb_gemm_device.h"

namespace mb {

// Cache policy of the C stores: written through the XCD's L2 (device scope,
// sc1). The tiles of a round end together, and lines left dirty would wait in
// the L2 for the flush at the kernel's end. 2048^3 (us): BF16 20.96 -> 19.77,
// MXFP4 10.43 -> 9.24; 1024^3 BF16 5.51 -> 5.13. Where an output of many rounds
// has rows of partial 128-byte lines, which stores then share, plain stores are
// better (BF16 7000x9001x1040 179, with sc1 236), as they are for the 256x256
// kernels' 64-byte stores (FP8 5000x3000x4112 61.5, with sc1 68.3).
// Non-temporal stores gain as much at 2048^3, but MXFP4 4096^3 on 256x128 tiles
// takes 50.4 with them, 45.8 with sc1, 47.9 plain.
// Order: such outputs store a row's pieces one after the other, so that shared
// lines are completed at once (the 179, column blocks outermost: 197); in few
// rounds, column blocks outermost is better (2048^3 BF16 20.0, rows 21.5).
// "Many" is more than two rounds of the chip for the 64x64 and the four-stage
// 128x128 tile: over 250 ragged shapes of 5 formats, plain rows against sc1
// columns take up to 14% more below one round, from 13% more to 18% less from
// one to two, 4.1% less on average from two to four and 8% less (never over 1%
// more) beyond; outputs past the memory-side cache gain most (FP64 7072x5406x4 on
// 64x64 tiles 146 -> 55).
constexpr int kStoreThrough = 16;

template <class Op, int BM, int BN, int STAGES>
struct RingTile {
  static constexpr int ROWB = 128;                     // bytes of K per row and step
  static constexpr int GROUPS = 64 / Op::M;            // lanes sharing a row, split over K
  static constexpr int CHUNKS = 8 / GROUPS;            // 16-byte chunks per lane and row block
  static constexpr int WM = BM / 2, WN = BN / 2;       // four waves in a 2x2 grid
  static constexpr int FM = WM / Op::M, FN = WN / Op::M;
  static constexpr int PER = ROWB / MfmaGeometry<Op>::K_BYTES;  // instructions per block and step
  static constexpr int DMA_A = BM / 32, DMA_B = BN / 32, DMA_S = Op::SCALED ? 1 : 0;
  static constexpr int DMAS = DMA_A + DMA_B + DMA_S;   // per wave and step
  static constexpr int OPERANDS = (BM + BN) * ROWB;
  static constexpr int SCALES_A = BM > 128 ? 2048 : 1024;  // bytes: 8 per row, in whole DMAs
  static constexpr int STAGE = OPERANDS + (Op::SCALED ? SCALES_A + 1024 : 0);
  // The tiles that large outputs run on; the others are mostly launched for few rounds.
  static constexpr bool MANY_ROUNDS = BM > 128 || STAGES == 2;
  static constexpr int MFMAS = FM * FN * PER, READS = (FM + FN) * CHUNKS;
  static_assert(Op::M == Op::N && WM % Op::M == 0 && WN % Op::N == 0, "whole instructions per wave");
  static_assert(BM % 64 == 0 && BN % 64 == 0 && BM <= 256 && BN <= 128, "whole DMAs per wave; scale rows per stage");
  static_assert(STAGES >= 2 && (STAGES - 1) * DMAS < 64, "vmcnt counts the DMAs in flight");
  static constexpr int RESIDENT = 160 * 1024 / (STAGES * STAGE);  // workgroups a CU's LDS holds
  static_assert(RESIDENT >= 1, "LDS");
};

// C = A . B^T over K steps of 128 bytes per row, for every instruction of
// mb_mfma.h in its widest form (32x32; 16x16 for FP64).
//
// LDS: a ring of STAGES stages, each [BM rows of A][BN rows of B] x 128 bytes
// (then, for MXFP4, 8 scale bytes per row of A and of B) with the XOR
// swizzle of the 256x256 kernels: row r holds its 16-byte chunk c at
// r*128 + ((c ^ ((r >> 1) & 7)) << 4). LDS-DMA loads fill it; wave w moves rows
// w*BM/4 .. of A and w*BN/4 .. of B, 8 rows an instruction.
//
// Fragments: lane group g of a row block holds chunks g, g + GROUPS, .. of its
// row. Instructions of 16-byte operands take one chunk each, in K order; FP8
// takes two, FP32 one float and FP64 one double of them, the same K permutation
// for A and B. Two register sets: a step's MFMAs use one while the next step's
// fragments are read into the other.
//
// Step kt: wait until this wave's DMAs of step kt+1 have landed; barrier (so
// everyone's have, and every read of stage kt % STAGES, made during step kt-1,
// has ended); then, spread over the step's MFMAs, the fragment reads of step
// kt+1 and the DMAs of step kt+STAGES into stage kt % STAGES. A stage is thus
// refilled STAGES-1 steps before it is needed.
//
// What bounds it: the matrix cores for FP32 and FP64 (a step's MFMAs take 4096
// cycles at 128x128; FP64 2048^3 runs at 89% of their rate, a few hundred cycles
// a step go to its barrier). For the narrower formats they take 512, and a full
// chip measures 0.43-0.48 us (about 1030 cycles) a step: 32 KiB per CU, 19 TB/s
// from the L2s, of which about 4 TB/s cross the fabric at 2048^3 (50 MB of reads:
// each XCD fetches its own copy of its 12 panels). Splitting a step's K over the waves, which
// halves the LDS reads (64 KiB, 512 cycles), takes 4% off a step and adds a
// final sum: 18.9 -> 19.8 us at 2048^3. 256x128 moves 25% less per output;
// 64x64 moves twice as much, but fills the chip from 1024^3 on. Stages: 128x128
// needs 4 for its latency when
// a CU holds one tile (2048^3 BF16: 25.6 us with 2, 24 with 3, 20.9 with 4, 23
// with 5) and 2 when it can hold a pair, whose prologues and stores overlap
// (4096^3: 118 us with 2, 129 with 4); 64x64 gains nothing from more than 3
// (1024^3: 5.6 us with 3, 5.8 with 5, 6.2 with 8).
//
// Measured against the largest tile it replaces (us): BF16 256^3 10.6 -> 3.1,
// 1024^3 22.3 -> 5.6, 2048^3 39.3 -> 20.4, 2560^3 47.9 -> 34.1; FP16
// 1000x744x1000 16.8 -> 5.5; MXFP4 2048^3
// 19.4 -> 10.2; FP32 1024^3 226 -> 22; FP64 2048^3 456 -> 248.
//
// Any shape: rows past M or N, chunks past K and steps past the last get an
// out-of-range offset, which the buffer bounds check turns into zeros (also in
// LDS) without a memory access, so every wave issues the same DMAs in every
// step and vmcnt counts them; stores past the edge are dropped the same way.
// MXFP4 scale bytes past K are masked to 0 (2^-127) in registers: whatever the
// caller's padding holds, NaN included, never meets the zeroed operands.
template <class Op, int BM, int BN, int STAGES>
__global__ void __launch_bounds__(256)
    gemm_ring_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, const uint8_t* __restrict__ SA,
                     const uint8_t* __restrict__ SB, typename Op::Out* __restrict__ C, int M, int N, int K,
                     int group_m) {
#if defined(__HIP_DEVICE_COMPILE__)
  using T = RingTile<Op, BM, BN, STAGES>;
  constexpr int ROWB = T::ROWB, FM = T::FM, FN = T::FN, CH = T::CHUNKS;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * T::STAGE];
  if (K < 0) lds[threadIdx.x] = 0;  // keeps DMA-written reads live; never executed

  int tile_m, tile_n;
  band_tile_any((static_cast<uint32_t>(M) + BM - 1) / BM, (static_cast<uint32_t>(N) + BN - 1) / BN, group_m, tile_m,
                tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int row_bytes = K * Op::ELEM_BITS / 8;
  const int k_steps = (row_bytes + ROWB - 1) / ROWB;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t ra =
      buffer_rsrc(A + static_cast<int64_t>(m0) * row_bytes, min(BM, M - m0) * row_bytes);
  const __amdgpu_buffer_rsrc_t rb =
      buffer_rsrc(B + static_cast<int64_t>(n0) * row_bytes, min(BN, N - n0) * row_bytes);
  // Lane l of a DMA fills row l/8, physical chunk l%8, from the logical chunk
  // stored there; rows 8 apart alternate between two swizzles. A chunk lies
  // inside its row in step kt while kt * 128 < its limit.
  const int drow = lane >> 3;
  const int chunk0 = (lane & 7) ^ (drow >> 1), chunk1 = chunk0 ^ 4;
  const int limit0 = row_bytes - 16 * chunk0, limit1 = row_bytes - 16 * chunk1;
  int va[T::DMA_A], vb[T::DMA_B];
#pragma unroll
  for (int i = 0; i < T::DMA_A; ++i)
    va[i] = (wave * (BM / 4) + 8 * i + drow) * row_bytes + 16 * ((i & 1) ? chunk1 : chunk0);
#pragma unroll
  for (int i = 0; i < T::DMA_B; ++i)
    vb[i] = (wave * (BN / 4) + 8 * i + drow) * row_bytes + 16 * ((i & 1) ? chunk1 : chunk0);
  const uint32_t lds_base =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds));
  const int scale_half = BM > 128 && !(wave & 1) ? wave >> 1 : 0;
  const int scale_rows = (wave & 1) ? N : M;
  const int scale_row0 = scale_first_row(BM, wave, m0, n0);
  const __amdgpu_buffer_rsrc_t rs =
      (wave & 1) ? buffer_rsrc(SB, Op::SCALED ? k_steps * N * 8 : 0) : buffer_rsrc(SA, Op::SCALED ? k_steps * M * 8 : 0);

  // DMA i of step kt into the stage at byte offset `stage`.
  auto dma = [&](auto i_c, int kt, uint32_t stage) __attribute__((always_inline)) {
    constexpr int i = decltype(i_c)::value;
    const int kb = kt * ROWB;
    const int soffset = __builtin_amdgcn_readfirstlane(kt < k_steps ? kb : 0);  // an offset past num_records would wrap the bounds check
    if constexpr (i < T::DMA_A) {
      dma16(ra, kb < ((i & 1) ? limit1 : limit0) ? va[i] : kOutOfRange, soffset,
            lds_base + (wave * (BM / 4) + 8 * i) * ROWB, stage);
    } else if constexpr (i < T::DMA_A + T::DMA_B) {
      constexpr int j = i - T::DMA_A;
      dma16(rb, kb < ((j & 1) ? limit1 : limit0) ? vb[j] : kOutOfRange, soffset,
            lds_base + (BM + wave * (BN / 4) + 8 * j) * ROWB, stage);
    } else {
      const DmaOffsets at = scale_offsets(kt, k_steps, scale_rows, scale_row0, lane);
      dma16(rs, at.lane, __builtin_amdgcn_readfirstlane(at.scalar),
            lds_base + T::OPERANDS + ((wave & 1) ? T::SCALES_A : scale_half * 1024), stage);
    }
  };

  const int wm = wave & 1, wn = wave >> 1;
  const int lrow = lane % Op::M, lgroup = lane / Op::M;
  const int swizzle = ((lrow >> 1) & 7) ^ lgroup;
  // Chunk i of the lane's fragment: its base with address bits 4..6 XORed;
  // stage and row block offsets are multiples of 1 KiB and add to it.
  const uint32_t la = (wm * T::WM + lrow) * ROWB + (swizzle << 4);
  const uint32_t lb = (BM + wn * T::WN + lrow) * ROWB + (swizzle << 4);
  struct Set {
    i32x4 a[FM][CH], b[FN][CH];
    uint32_t sa[FM], sb[FN];
  };
  auto read = [&](auto r_c, Set& set, uint32_t stage) __attribute__((always_inline)) {
    constexpr int r = decltype(r_c)::value, c = r / (FM + FN), f = r % (FM + FN);
    if constexpr (f < FM)
      set.a[f][c] = *reinterpret_cast<const i32x4*>(lds + stage + (la ^ (c * T::GROUPS << 4)) + f * Op::M * ROWB);
    else
      set.b[f - FM][c] =
          *reinterpret_cast<const i32x4*>(lds + stage + (lb ^ (c * T::GROUPS << 4)) + (f - FM) * Op::M * ROWB);
  };
  // One dword per row block with the lane's four scale bytes (K groups lgroup,
  // 2 + lgroup, ..: instruction p uses byte p); bytes past K are masked.
  const uint32_t pick = 0x06040200u + 0x01010101u * static_cast<uint32_t>(lgroup);
  uint32_t tail_mask = 0;
  if constexpr (Op::SCALED) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
      if (((k_steps - 1) * 8 + 2 * p + lgroup) * 32 < K) tail_mask |= 0xffu << (8 * p);
  }
  auto read_scales = [&](Set& set, int kt, uint32_t stage) __attribute__((always_inline)) {
    const uint32_t mask = kt == k_steps - 1 ? tail_mask : 0xffffffffu;
    auto scale = [&](int row) __attribute__((always_inline)) {
      const i32x2 v = *reinterpret_cast<const i32x2*>(lds + stage + T::OPERANDS + row * 8);
      return __builtin_amdgcn_perm(static_cast<uint32_t>(v[1]), static_cast<uint32_t>(v[0]), pick) & mask;
    };
#pragma unroll
    for (int f = 0; f < FM; ++f) set.sa[f] = scale(wm * T::WM + f * Op::M + lrow);
#pragma unroll
    for (int f = 0; f < FN; ++f) set.sb[f] = scale(T::SCALES_A / 8 + wn * T::WN + f * Op::M + lrow);
  };

  typename Op::Acc acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = typename Op::Acc{};
  // FP64 accumulates in place through mma_tied (the compiler copies the 16x16
  // accumulators otherwise), under its hazard rules.
  auto fence = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc_hazard_fence(acc[i][j]);
  };
  auto mma = [&](auto q_c, const Set& set) __attribute__((always_inline)) {
    constexpr int q = decltype(q_c)::value, p = q / (FM * FN), i = q % (FM * FN) / FN, j = q % FN;
    const i32x4(&a)[CH] = set.a[i];
    const i32x4(&b)[CH] = set.b[j];
    if constexpr (Op::SCALED) {
      acc[i][j] = Op::template mma_byte<p>(a[p], b[p], acc[i][j], set.sa[i], set.sb[j]);
    } else if constexpr (Op::LANE_BYTES == 16) {
      acc[i][j] = Op::mma(a[p], b[p], acc[i][j], 0, 0);
    } else if constexpr (Op::LANE_BYTES == 32) {
      acc[i][j] = Op::mma(__builtin_shufflevector(a[2 * p], a[2 * p + 1], 0, 1, 2, 3, 4, 5, 6, 7),
                          __builtin_shufflevector(b[2 * p], b[2 * p + 1], 0, 1, 2, 3, 4, 5, 6, 7), acc[i][j], 0, 0);
    } else if constexpr (Op::LANE_BYTES == 8) {
      typedef double f64x2 __attribute__((ext_vector_type(2)));
      Op::mma_tied(__builtin_bit_cast(f64x2, a[p / 2])[p % 2], __builtin_bit_cast(f64x2, b[p / 2])[p % 2], acc[i][j]);
    } else {
      acc[i][j] = Op::mma(__builtin_bit_cast(f32x4, a[p / 4])[p % 4], __builtin_bit_cast(f32x4, b[p / 4])[p % 4],
                          acc[i][j], 0, 0);
    }
  };

  // Prologue: steps 0 .. STAGES-1 in flight, step 0's fragments in set 0.
  static_for<0, STAGES>([&](auto s_c) __attribute__((always_inline)) {
    static_for<0, T::DMAS>([&](auto i_c) __attribute__((always_inline)) {
      dma(i_c, decltype(s_c)::value, decltype(s_c)::value * T::STAGE);
    });
  });
  __builtin_amdgcn_s_waitcnt(vmcnt_only((STAGES - 1) * T::DMAS));
  lds_barrier();
  Set set0, set1;
  static_for<0, T::READS>([&](auto r_c) __attribute__((always_inline)) { read(r_c, set0, 0); });
  if constexpr (Op::SCALED) read_scales(set0, 0, 0);

  uint32_t stage = 0;  // byte offset of step kt's stage
  auto step = [&](int kt, const Set& set, Set& next) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(vmcnt_only((STAGES - 2) * T::DMAS));
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t next_stage = stage == (STAGES - 1) * T::STAGE ? 0 : stage + T::STAGE;
    if constexpr (Op::SCALED) read_scales(next, kt + 1, next_stage);
    // Reads are done by three quarters of the MFMAs, so the next barrier does
    // not wait for them; the DMAs are spread over all.
    constexpr int NQ = T::MFMAS, NR = T::READS, READ_Q = NQ - NQ / 4;
    static_for<0, NQ>([&](auto q_c) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value;
      constexpr int r0 = q < READ_Q ? q * NR / READ_Q : NR, r1 = q + 1 < READ_Q ? (q + 1) * NR / READ_Q : NR;
      static_for<r0, r1>([&](auto r_c) __attribute__((always_inline)) { read(r_c, next, next_stage); });
      static_for<q * T::DMAS / NQ, (q + 1) * T::DMAS / NQ>(
          [&](auto i_c) __attribute__((always_inline)) { dma(i_c, kt + STAGES, stage); });
      mma(q_c, set);
      __builtin_amdgcn_sched_barrier(0);
    });
    stage = next_stage;
  };
  if constexpr (Op::LANE_BYTES == 8) fence();
  int kt = 0;
  for (; kt + 1 < k_steps; kt += 2) {
    step(kt, set0, set1);
    step(kt + 1, set1, set0);
  }
  if (kt < k_steps) step(kt, set0, set1);
  if constexpr (Op::LANE_BYTES == 8) fence();
  __builtin_amdgcn_s_waitcnt(vmcnt_only(0));  // no DMA of a step past the last may land in a later workgroup's LDS

  // Rows past M lie past num_records; columns past N get an out-of-range offset.
  constexpr int ES = sizeof(typename Op::Out);
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      C + static_cast<int64_t>(m0) * N + n0, (short)0, min(BM, M - m0) * N * ES - n0 * ES, kBufferWord3);
  auto store = [&](int i, int j, int r, auto policy_c) __attribute__((always_inline)) {
    constexpr int policy = decltype(policy_c)::value;
    const int col = wn * T::WN + j * Op::N + lane % Op::N;
    const int offset = ((wm * T::WM + i * Op::M + Op::out_row(lane, r)) * N + col) * ES;
    const int at = n0 + col < N ? offset : kOutOfRange;
    const typename Op::Out value = acc[i][j][r];
    if constexpr (ES == 8)
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, value), rc, at, 0, policy);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, value), rc, at, 0, policy);
  };
  auto store_rows = [&](auto policy_c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < Op::ACC_REGS; ++r)
#pragma unroll
        for (int j = 0; j < FN; ++j) store(i, j, r, policy_c);
  };
  const bool whole_lines = (static_cast<int64_t>(N) * ES | reinterpret_cast<intptr_t>(C)) % 128 == 0;
  if (!whole_lines && (T::MANY_ROUNDS || gridDim.x > 2 * 256 * T::RESIDENT)) {
    store_rows(std::integral_constant<int, 0>{});
  } else if constexpr (T::MANY_ROUNDS) {
    store_rows(std::integral_constant<int, kStoreThrough>{});
  } else {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < Op::ACC_REGS; ++r) store(i, j, r, std::integral_constant<int, kStoreThrough>{});
  }
#endif
}

}  // namespace mb
