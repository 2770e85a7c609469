"""mb_copy where source or destination lie off the 16-byte grid or the length off it: every byte of the range
arrives, nothing outside it is written, at lengths around one vector, the 128-byte head and a workgroup."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1, 15, 16, 17, 111, 112, 113, 127, 128, 143, 144, 145, 1000, 64 * 16 + 127, 256 * 16 * 4 + 5, (1 << 20) + 3]


@pytest.mark.parametrize("flags", [0, 1, 3])
@pytest.mark.parametrize("src_offset,dst_offset", [(0, 0), (4, 4), (1, 1), (0, 2), (6, 0), (3, 13), (0, 16), (8, 127)])
def test_every_byte_and_nothing_else(gpu, flags, src_offset, dst_offset):
    import torch

    from triton_chip_benchmarks_amd import _native

    raw = torch.randint(0, 256, ((1 << 20) + 512,), dtype=torch.uint8, device="cuda")
    want = raw.cpu().numpy()
    for count in LENGTHS:
        for threads, vectors, grid in ((64, 1, 0), (256, 4, 0), (1024, 16, 2)):
            print(f"copy {count} bytes +{src_offset} -> +{dst_offset} threads={threads} vectors={vectors} grid={grid} "
                  f"flags={flags}", flush=True)
            out = torch.full_like(raw, 0x5A)
            _native.call("mb_copy", raw.data_ptr() + src_offset, out.data_ptr() + dst_offset, count, threads, vectors,
                         grid, flags, _native.stream_handle())
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            assert np.array_equal(got[dst_offset:dst_offset + count], want[src_offset:src_offset + count])
            assert (got[:dst_offset] == 0x5A).all() and (got[dst_offset + count:] == 0x5A).all()
