"""Every byte that the ring GEMM kernel's scale DMAs read lies in the scale buffer, over shapes, on the CPU.

The kernel's own offset functions are compiled for the host. The bounds check is applied as the hardware does it: a
dword passes when its vector offset is below num_records minus the scalar offset, in unsigned 32-bit arithmetic.
"""

from pathlib import Path
import shutil
import subprocess

import pytest

CSRC = Path(__file__).resolve().parent.parent / "triton_chip_benchmarks_amd" / "csrc"
PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include "mb_gemm_offsets.h"

int main() {
  long outside = 0, wrapped = 0, missing = 0;
  const int stages = 4;
  for (int tile : {64, 128, 256})
    for (int rows = 1; rows <= 777; ++rows)
      for (int k_steps : {1, 2, 5})
        for (int row0 = 0; row0 < rows; row0 += tile)
          for (int wave = 0; wave < 4; ++wave) {
            const uint32_t size = k_steps * rows * 8;
            // A's rows through m0 for waves 0 and 2, B's (tiles of up to 128) through n0 for the others.
            if ((wave & 1) && tile > 128) continue;
            const int first = mb::scale_first_row(tile, wave, row0, row0);
            for (int kt = 0; kt < k_steps + stages; ++kt)
              for (int lane = 0; lane < 64; ++lane) {
                const mb::DmaOffsets at = mb::scale_offsets(kt, k_steps, rows, first, lane);
                if (static_cast<uint32_t>(at.scalar) > size) ++wrapped;
                for (int dword = 0; dword < 4; ++dword) {
                  const uint32_t vector = static_cast<uint32_t>(at.lane) + 4 * dword;
                  const bool read = vector < size - static_cast<uint32_t>(at.scalar);
                  if (read && static_cast<uint64_t>(vector) + at.scalar >= size) ++outside;
                  const int row = first + lane * 2 + dword / 2;  // 8 bytes a row
                  if (kt < k_steps && row < rows &&
                      (!read || vector + at.scalar != (static_cast<uint32_t>(kt) * rows + row) * 8 + dword % 2 * 4))
                    ++missing;
                }
              }
          }
  std::printf("%ld %ld %ld\n", outside, wrapped, missing);
}
"""


def test_scale_dmas_read_inside_the_scale_buffer(tmp_path):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("g++ is not installed")
    (tmp_path / "check.cpp").write_text(PROGRAM)
    subprocess.run([compiler, "-O2", "-std=c++17", f"-I{CSRC}", str(tmp_path / "check.cpp"), "-o",
                    str(tmp_path / "check")], check=True)
    outside, wrapped, missing = map(int, subprocess.run([str(tmp_path / "check")], check=True, capture_output=True,
                                                         text=True).stdout.split())
    assert (outside, wrapped, missing) == (0, 0, 0)
