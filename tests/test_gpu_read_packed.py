"""mb_read_sum where its kernels change: segments packed into a wave, last chunks, clipped segments and
misaligned sources, for every segment size."""

import numpy as np
import pytest

from oracle import memory

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype_name", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("block", [64, 128, 256, 512, 1024, 2048, 4096, 8192, 65536])
@pytest.mark.parametrize("whole,clipped", [(0, 1), (1, 0), (31, 0), (33, 17), (70, -1)])
def test_every_segment_size_sums_exactly(gpu, dtype_name, block, whole, clipped):
    """Integers of magnitude up to 2 sum exactly in fp32 in any order, so a dropped, doubled or misplaced
    element shows; the source starts on and one element off the 16-byte grid, a guard follows the sink."""
    import torch

    from triton_chip_benchmarks_amd.bench_bandwidth import launch_read, torch_dtype

    elements = whole * block + (clipped % block)
    segments = -(-elements // block)
    values = torch.randint(-2, 3, (elements + 1,), device="cuda", generator=torch.Generator("cuda").manual_seed(block))
    values = values.to(torch_dtype(dtype_name))
    for offset in (0, 1):
        src = values[offset:offset + elements]
        print(f"read {dtype_name} block={block} elements={elements} offset={offset}", flush=True)
        sink = torch.full((segments + 64,), -7.0, device="cuda")
        launch_read(src, sink, block, 256)
        torch.cuda.synchronize()
        got = sink.cpu().numpy()
        assert np.array_equal(got[:segments].astype(np.float64), memory.block_sums(src.float().cpu().numpy(), block))
        assert (got[segments:] == -7.0).all()


@pytest.mark.parametrize("dtype_name,block,elements", [("fp32", 1024, (1 << 27) + (1 << 20) + 5),
                                                       ("bf16", 64, (1 << 28) + (1 << 21) + 3)])
def test_past_the_wave_count_of_single_loads(gpu, dtype_name, block, elements):
    """More than 131072 waves: each keeps one load in flight."""
    import torch

    from triton_chip_benchmarks_amd.bench_bandwidth import check_read, launch_read, torch_dtype

    print(f"read {dtype_name} block={block} elements={elements}", flush=True)
    src = torch.empty(elements, device="cuda", dtype=torch_dtype(dtype_name)).uniform_(-1, 1)
    sink = torch.full((-(-elements // block),), float("nan"), device="cuda")
    launch_read(src, sink, block, 256)
    torch.cuda.synchronize()
    check_read(src, sink, block)
