// Buffer offsets of the GEMM kernels' LDS-DMA loads. Plain C++, so that the
// host can check them over shapes.
#pragma once

namespace mb {

// A byte offset past every buffer resource (num_records stays below 2^31):
// loads from it give zeros, stores to it are dropped.
constexpr int kOutOfRange = static_cast<int>(0x80000000u);

// Vector offset of a lane and scalar offset of one LDS-DMA load. The bounds
// check compares the vector offset with the buffer's size less the scalar
// offset, which therefore must not exceed it: the difference would wrap and
// every lane pass.
struct DmaOffsets {
  int lane, scalar;
};

// First row of the 128 whose scales wave `wave` of a tile at (m0, n0) moves:
// waves 0 and 2 move A's, 1 and 3 B's; tiles of up to 128 rows are moved twice,
// so that every wave has the same DMA count.
constexpr int scale_first_row(int tile_rows, int wave, int m0, int n0) {
  return (wave & 1) ? n0 : tile_rows > 128 && wave == 2 ? m0 + 128 : m0;
}

// The scales ([k_steps][rows][8] bytes) of rows first .. first + 127 in step kt.
// Nothing where a tile's second 128 rows all lie past the last one: in the last
// step the scalar offset would exceed the buffer.
constexpr DmaOffsets scale_offsets(int kt, int k_steps, int rows, int first, int lane) {
  return kt < k_steps && first < rows ? DmaOffsets{lane * 16, (kt * rows + first) * 8} : DmaOffsets{kOutOfRange, 0};
}

}  // namespace mb
