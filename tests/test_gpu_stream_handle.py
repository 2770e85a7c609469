"""stream_handle: the raw handle of the stream that torch would use, on every thread and inside stream contexts."""

import threading

import pytest

pytestmark = pytest.mark.gpu


def test_handle_follows_the_current_stream(gpu):
    import torch

    from triton_chip_benchmarks_amd import _native

    def expected():
        return torch.cuda.current_stream().cuda_stream or None

    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    assert _native.stream_handle() == expected()
    with torch.cuda.stream(side):
        assert _native.stream_handle() == expected() == side.cuda_stream
        with torch.cuda.stream(other):
            assert _native.stream_handle() == other.cuda_stream
        assert _native.stream_handle() == side.cuda_stream
        seen = []  # a new thread starts on its own current stream, the default one
        thread = threading.Thread(target=lambda: seen.append((_native.stream_handle(), expected())))
        thread.start()
        thread.join()
        assert seen[0][0] == seen[0][1]
        assert _native.stream_handle(other) == other.cuda_stream
    assert _native.stream_handle() == expected()


def test_a_launch_on_a_side_stream_is_captured_there(gpu):
    """A copy issued inside a capture lands in the graph and runs on each replay."""
    import torch

    from triton_chip_benchmarks_amd.bench_bandwidth import launch_copy

    src = torch.zeros(1000, device="cuda")
    dst = torch.full_like(src, -1.0)
    launch_copy(src, dst, 256, 1, 0, "off")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch_copy(src, dst, 256, 1, 0, "off")
    for value in (1.0, 2.0, 3.0):
        src.fill_(value)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert bool((dst == value).all())
