"""The kernel that a GEMM row names is the one its launches run, on the CPU (launches recorded, not made)."""

from pathlib import Path
import sys
from types import SimpleNamespace

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent))

import bench  # noqa: E402
from triton_chip_benchmarks_amd import _native, crosscheck, gemm  # noqa: E402

SIZE = 512  # where smaller tiles than the largest run


@pytest.fixture
def on_cpu(monkeypatch):
    inputs = gemm.gemm_inputs
    monkeypatch.setattr(gemm, "gemm_inputs", lambda dtype, m, n, k, device, seed: inputs(dtype, m, n, k, "cpu", seed))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: None)


def _launched(dtype):
    config = max(_native.gemm_configs(dtype), key=lambda c: c["tile_m"] * c["tile_n"])
    return _native.gemm_launched_kernel(dtype, config, SIZE, SIZE, SIZE)


@pytest.mark.parametrize("dtype", ["bf16", "fp8", "fp64", "fp4"])
def test_bench_gemm_rows_name_the_launched_kernel_and_its_tile(on_cpu, dtype):
    workload = bench.GemmWorkload(torch, 256, "gemm", dtype, SIZE)
    assert workload.kernel == _launched(dtype)
    assert workload.config["tile"] == workload.kernel.split("_")[2]


def test_crosscheck_rows_name_the_launched_kernel(on_cpu, monkeypatch):
    monkeypatch.setattr(_native, "gemm", lambda dtype, config, a, b, c, m, n, k, *scales: c.zero_())
    monkeypatch.setattr(crosscheck, "_library_gemm", lambda *arguments: None)
    monkeypatch.setattr(crosscheck, "measure", lambda run, args: {"min_ms": 1.0, "median_ms": 1.0})
    rows = crosscheck.gemm_rows(SimpleNamespace(seed=0), ["bf16", "fp8", "fp64", "fp32"], SIZE, SIZE, SIZE)
    ours = {row["dtype"]: row["kernel"] for row in rows if row["path"] == "mb_gemm"}
    assert ours == {dtype: _launched(dtype) for dtype in ("bf16", "fp8", "fp64", "fp32")}
