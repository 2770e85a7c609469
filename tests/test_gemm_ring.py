"""The GEMM kernels of any shape (the ring and the ragged 256x256 ones) at the edges of their tiles, K steps and dispatch, against oracle.tensor.

Operands are exact lattices (FP64: N(0,1) within its tolerance), so the
comparison is exact. The shapes reach every such kernel of every format with M
and N off its tile and K off its 128-byte step (a CPU test pins that).
"""

import numpy as np
import pytest

from oracle import tensor as ot
from test_gpu_gemm import FORMATS, _assert_matches, _configs, _run_gemm, _scale_blocks

CHUNK = {"bf16": 8, "fp16": 8, "fp32": 4, "fp64": 2, "int8": 16, "fp8": 16, "fp4": 32}  # elements per 16 bytes
# (M, N, 16-byte chunks of K): one element, one step exactly, tails in M, N and K, odd and even step counts;
# then one shape per larger tile.
SHAPES = [(1, 1, 1), (64, 64, 8), (65, 63, 9), (130, 70, 23), (192, 128, 16), (2040, 2035, 33), (2040, 2035, 145),
          (2047, 2049, 9), (2600, 2500, 161), (3800, 3900, 161)]


class _Scales:
    """Stands in for an aligned device tensor where only the pointer matters."""

    def data_ptr(self):
        return 4096

    def numel(self):
        return 1

    def element_size(self):
        return 1


def _launched(dtype, config, m, n, k, **options):
    from triton_chip_benchmarks_amd import _native

    scales = (_Scales(), _Scales()) if dtype == "fp4" else (None, None)
    return _native.gemm_launched_kernel(dtype, config, m, n, k, *scales, **options)


@pytest.mark.parametrize("dtype", FORMATS)
def test_shapes_reach_every_kernel_of_any_shape(dtype):
    from triton_chip_benchmarks_amd import _native

    prefix = _native.gemm_kernel_name(dtype, _configs(dtype)[0]).rsplit("_", 1)[0] + "_"
    wanted = {name for name in _native.kernel_names()
              if name.startswith(prefix) and not name.endswith("_checked")
              and ("_256x256x" not in name or name.endswith("_ragged")) and name != "gemm_f64_256x128x16"}
    seen = {_launched(dtype, config, m, n, chunks * CHUNK[dtype])
            for config in _configs(dtype) for m, n, chunks in SHAPES}
    assert wanted <= seen, wanted - seen


@pytest.mark.parametrize("dtype", FORMATS)
def test_a_launch_never_exceeds_the_requested_tile(dtype):
    """Whatever the shape, the launched kernel's tile fits inside the requested one, and rows too long for
    32-bit offsets, one of the checked kernel's cases, go to it."""
    for config in _configs(dtype):
        for m, n, k in [(1, 1, 256), (300, 5000, 512), (4096, 4096, 4096), (8192, 256, 1024)]:
            tile = _launched(dtype, config, m, n, k).split("_")[2]
            tile_m, tile_n, _ = (int(x) for x in tile.split("x"))
            assert tile_m <= config["tile_m"] and tile_n <= config["tile_n"], (config, m, n, k, tile)
        assert _launched(dtype, config, 64, 64, (1 << 22) * CHUNK[dtype]).endswith("_checked")


@pytest.mark.parametrize("dtype,m,n,k,name", [("fp32", 8192, 8192, 8192, "gemm_f32_256x256x32"),
                                              ("fp32", 4096, 4096, 4096, "gemm_f32_256x256x32"),
                                              ("fp32", 3072, 10240, 7744, "gemm_f32_256x256x32"),
                                              ("fp64", 7936, 10240, 2304, "gemm_f64_256x128x16"),
                                              ("fp64", 512, 14848, 1856, "gemm_f64_256x128x16"),
                                              ("fp32", 2048, 2048, 2048, "gemm_f32_128x128x32"),
                                              ("fp32", 1536, 7936, 10944, "gemm_f32_128x128x32"),
                                              ("fp64", 2048, 2048, 2048, "gemm_f64_128x128x16"),
                                              ("fp4", 8704, 256, 3584, "gemm_mxfp4_128x128x256"),
                                              ("fp4", 1024, 2816, 2048, "gemm_mxfp4_128x128x256")])
def test_shapes_take_the_kernel_measured_fastest(dtype, m, n, k, name):
    """Smaller tiles are 3 to 6% slower at the first five; at the others larger ones leave CUs idle and smaller ones
    move more operands (64x64 is 29% and 44% slower at the MXFP4 shapes)."""
    assert _launched(dtype, max(_configs(dtype), key=lambda c: c["tile_m"] * c["tile_n"]), m, n, k) == name


@pytest.mark.parametrize("dtype", FORMATS)
def test_an_exact_tile_launch_runs_that_tile_or_is_refused(dtype):
    """exact_tile: the kernel's tile is the configured one whatever else would be faster; where no kernel of the tile
    takes the shape the call is refused."""
    from triton_chip_benchmarks_amd import _native

    step = 8 * CHUNK[dtype]
    for config in _configs(dtype):
        for m, n, k in [(512, 768, 4 * step), (2048, 2048, 16 * step), (300, 200, CHUNK[dtype])]:
            takes_any = config["tile_m"] == config["tile_n"] == 128 or config["tile_n"] < 256 and \
                not (dtype == "fp64" and config["tile_m"] == 256) or dtype in ("bf16", "fp16", "int8", "fp8")
            if m == 300 and not takes_any:
                with pytest.raises(_native.NativeError, match="no kernel of tile"):
                    _launched(dtype, config, m, n, k, exact_tile=True)
                continue
            tile = _native.gemm_kernel_tile(_launched(dtype, config, m, n, k, exact_tile=True))
            assert {key: tile[key] for key in config} == config, (m, n, k)


@pytest.mark.parametrize("dtype", FORMATS)
@pytest.mark.parametrize("size", [256, 2048, 3000])
def test_the_gemm_sweep_times_every_tile_on_a_kernel_of_its_own(dtype, size):
    from triton_chip_benchmarks_amd import _native, gemm

    scales = (_Scales(), _Scales()) if dtype == "fp4" else (None, None)
    size = -(-size // 32) * 32
    launches = gemm.sweep_launches(dtype, _configs(dtype), size, scales)
    names = [name for _, _, name in launches]
    assert len(set(names)) == len(names)
    assert _launched(dtype, max(_configs(dtype), key=lambda c: c["tile_m"] * c["tile_n"]), size, size, size) in names
    for config, exact_tile, name in launches:
        tile = _native.gemm_kernel_tile(name)
        if exact_tile:
            assert (tile["tile_m"], tile["tile_n"]) == (config["tile_m"], config["tile_n"])
    if size == 2048:
        assert sum(exact for _, exact, _ in launches) == len(_configs(dtype))
    only = gemm.sweep_launches(dtype, _configs(dtype)[:1], size, scales, automatic=False)
    assert len(only) == 1


@pytest.mark.parametrize("dtype", FORMATS)
def test_very_tall_and_wide_shapes_get_a_grid_that_hip_takes(dtype):
    """A launch may have at most 2^32 - 1 work items, so 2^24 - 1 workgroups of 256: where 64x64 tiles are more, a
    larger tile runs; where every tile the caller allows is more, the call is refused."""
    from triton_chip_benchmarks_amd import _native

    config = max(_configs(dtype), key=lambda c: c["tile_m"] * c["tile_n"])
    for m, n in [(2**30, 1), (2**30 + 1, 64), (1, 2**30), (70, 2**29), (2**20, 2**10), (2**30 - 64, 1)]:
        name = _launched(dtype, config, m, n, CHUNK[dtype])
        tile_m, tile_n, _ = (int(x) for x in name.split("_")[2].split("x"))
        assert -(-m // tile_m) * -(-n // tile_n) * 256 < 2**32, (m, n, name)
    small = {**config, "tile_m": 128, "tile_n": 128}
    with pytest.raises(_native.NativeError, match="too many tiles"):
        _launched(dtype, small, 2**31 - 1, 1, CHUNK[dtype])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", FORMATS)
@pytest.mark.parametrize("m,n,chunks", SHAPES)
def test_kernels_of_any_shape_match_oracle(gpu, dtype, m, n, chunks):
    k = chunks * CHUNK[dtype]
    rng = np.random.default_rng(m + n + k)
    for launched in sorted({_launched(dtype, config, m, n, k) for config in _configs(dtype)}):
        config = next(c for c in _configs(dtype) if _launched(dtype, c, m, n, k) == launched)
        print(f"gemm {dtype} {m}x{n}x{k} via {launched}", flush=True)
        got, a_values, b_values = _run_gemm(dtype, config, m, n, k, rng)
        _assert_matches(dtype, got, ot.gemm_reference(a_values, b_values.T))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", FORMATS)
def test_kernels_of_any_shape_write_only_c_and_read_nothing_past_their_operands(gpu, dtype):
    """C with guard rows and NaN (INT8: -3) bytes after A, B and the scales: a load past an edge that reached
    a product would show in C, a store past one in the guard."""
    import torch

    from triton_chip_benchmarks_amd import _native

    m, n, k = 67, 45, 11 * CHUNK[dtype]
    rng = np.random.default_rng(5)
    config = _configs(dtype)[0]
    scales = (None, None)
    if dtype == "fp4":
        codes = [rng.integers(0, 16, (rows, k), dtype=np.uint8) for rows in (m, n)]
        exponents = [rng.integers(126, 129, (rows, k // 32), dtype=np.uint8) for rows in (m, n)]
        values = [ot.e2m1_decode(c) * np.repeat(ot.e8m0_decode(s), 32, axis=1) for c, s in zip(codes, exponents)]
        blocks = [_scale_blocks(s) for s in exponents]
        for block in blocks:
            block[-1][:, (k // 32) % 8:] = 255  # the caller's padding: E8M0 NaN
        scales = tuple(torch.from_numpy(block).cuda() for block in blocks)
        a, b = (torch.from_numpy(ot.pack_e2m1(c)).cuda() for c in codes)
    else:
        _, *values, (_, a, b) = _run_gemm(dtype, config, m, n, k, rng, keep_device=True)
    poisoned = []
    for tensor in (a, b):
        poison = torch.full((tensor.numel() * tensor.element_size() + 4096,), 0xFF, dtype=torch.uint8, device="cuda")
        poison[:tensor.numel() * tensor.element_size()] = tensor.reshape(-1).view(torch.uint8)
        poisoned.append(poison)
    out = torch.int32 if dtype == "int8" else torch.float64 if dtype == "fp64" else torch.float32
    c = torch.full((m + 70, n), -3, dtype=out, device="cuda")
    _native.gemm(dtype, config, *poisoned, c, m, n, k, *scales)
    torch.cuda.synchronize()
    got = c.cpu().numpy().astype(np.float64)
    _assert_matches(dtype, got[:m], ot.gemm_reference(values[0], values[1].T))
    assert (got[m:] == -3).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tile", [("fp64", 64), ("fp64", 128), ("fp32", 128)])
@pytest.mark.parametrize("n", [3101, 3104])
def test_outputs_of_many_rounds_with_and_without_whole_lines(gpu, dtype, tile, n):
    """More than two rounds of the chip (2303 tiles of 64x64, 600 of 128x128), with rows of C that share 128-byte
    lines (n = 3101) and rows of whole lines: the stores take another order and cache policy. A request for 64x64
    tiles, or for 128x128, which FP32 answers with 64x64 here."""
    m, k = 3000, 3 * CHUNK[dtype]
    config = next(c for c in _configs(dtype) if c["tile_m"] == tile)
    exact = {"exact_tile": True} if dtype == "fp64" else {}
    name = _launched(dtype, config, m, n, k, **exact)
    assert name == {64: "gemm_f64_64x64x16", 128: "gemm_f64_128x128x16"}[tile] if exact else "gemm_f32_64x64x32"
    print(f"gemm {dtype} {m}x{n}x{k} via {name}", flush=True)
    got, a_values, b_values = _run_gemm(dtype, config, m, n, k, np.random.default_rng(n), **exact)
    _assert_matches(dtype, got, ot.gemm_reference(a_values, b_values.T))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp64", "fp8"])
def test_rows_past_the_32_bit_offsets_run_the_checked_kernel(gpu, dtype):
    """64 rows of 2^25 bytes are the first that a 64x64 tile cannot address with 31-bit offsets."""
    m, n, k = 3, 2, (1 << 21) * CHUNK[dtype]
    config = _configs(dtype)[0]
    assert _launched(dtype, config, m, n, k).endswith("_checked")
    print(f"gemm {dtype} {m}x{n}x{k} via {_launched(dtype, config, m, n, k)}", flush=True)
    got, a_values, b_values = _run_gemm(dtype, config, m, n, k, np.random.default_rng(3))
    reference = ot.gemm_reference(a_values, b_values.T)
    if dtype == "fp64":
        # Forward bound of K serial FMAs: K * 2^-53 * sum |a b|, here about 1e-9 of the sum.
        allowed = k * 2.0**-53 * ot.gemm_reference(np.abs(a_values), np.abs(b_values).T)
        assert np.all(np.abs(got - reference) <= allowed)
    else:
        _assert_matches(dtype, got, reference)


@pytest.mark.gpu
@pytest.mark.parametrize("offset,checked", [(1, True), (4, False)])
def test_mxfp4_scales_off_the_16_byte_grid(gpu, offset, checked):
    """Scales on a dword take the ring kernel's DMAs, byte-aligned ones the checked kernel."""
    import torch

    from triton_chip_benchmarks_amd import _native

    m, n, k = 70, 33, 544
    rng = np.random.default_rng(offset)
    codes = [rng.integers(0, 16, (rows, k), dtype=np.uint8) for rows in (m, n)]
    exponents = [rng.integers(126, 129, (rows, k // 32), dtype=np.uint8) for rows in (m, n)]
    values = [ot.e2m1_decode(c) * np.repeat(ot.e8m0_decode(s), 32, axis=1) for c, s in zip(codes, exponents)]
    scales = []
    for block in map(_scale_blocks, exponents):
        flat = torch.from_numpy(np.concatenate([np.zeros(offset, np.uint8), block.reshape(-1)])).cuda()
        scales.append(flat[offset:])
    config = _configs("fp4")[0]
    name = _native.gemm_launched_kernel("fp4", config, m, n, k, *scales)
    assert name.endswith("_checked") == checked
    print(f"gemm fp4 scale offset {offset} via {name}", flush=True)
    c = torch.full((m, n), float("nan"), device="cuda")
    _native.gemm("fp4", config, *(torch.from_numpy(ot.pack_e2m1(x)).cuda() for x in codes), c, m, n, k, *scales)
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy().astype(np.float64), ot.gemm_reference(values[0], values[1].T))


def _ring_kernels():
    """(name, stages, DMAs per wave and step) of every ring kernel."""
    from triton_chip_benchmarks_amd import _native, audit

    out = []
    for name in _native.kernel_names():
        symbol = audit.symbols().get(name, "")
        match = audit._GEMM_RING_RE.search(symbol)
        if match:
            _, bm, bn, stages = match.groups()
            out.append((name, int(stages), int(bm) // 32 + int(bn) // 32 + ("mxfp4" in name)))
    return out


def test_every_ring_kernel_stores_c_written_through_and_plain():
    """Written through the L2 (sc1), and plain for outputs of many rounds whose rows share lines, where the former
    is up to 2.6 times slower (FP64 7072x5406x4 on 64x64 tiles)."""
    from triton_chip_benchmarks_amd import audit

    for name, _, _ in _ring_kernels():
        stores = [line.split("//")[0] for line in audit.instructions(name)
                  if audit.mnemonic(line).startswith("buffer_store_dword")]
        assert {"sc1" in line for line in stores} == {True, False}, name


def test_ring_loops_wait_for_every_dma_and_every_read():
    """In the compiled loops, an LDS-DMA is retired by the waits within STAGES-1 barriers of its issue, after which
    its stage is read (one barrier less would be too few where the ring has a third stage), and every barrier,
    after which a stage just read is refilled, follows a wait for all LDS reads."""
    from test_audit import _dma_coverage_violations
    from triton_chip_benchmarks_amd import audit

    kernels = _ring_kernels()
    assert len(kernels) == 25
    for name, stages, dmas in kernels:
        body = audit.hot_loop(name)
        assert sum(line.rstrip().endswith(" lds") for line in body) == 2 * dmas, name
        assert sum(audit.mnemonic(line) == "s_barrier" for line in body) == 2, name
        assert _dma_coverage_violations(body, horizon=stages - 1) == [], name
        if stages > 2:
            assert _dma_coverage_violations(body, horizon=stages - 2), name
        unwaited = [line for line in body if not (audit.mnemonic(line) == "s_waitcnt" and "vmcnt" in line)]
        assert _dma_coverage_violations(unwaited, horizon=stages - 1), name
        # The reads of a step are all waited for before its closing barrier.
        pending = False
        for line in body + body:
            if audit.mnemonic(line).startswith("ds_read"):
                pending = True
            elif audit.mnemonic(line) == "s_waitcnt" and "lgkmcnt(0)" in line:
                pending = False
            elif audit.mnemonic(line) == "s_barrier":
                assert not pending, name


def test_lds_dmas_wait_a_state_after_the_write_of_m0():
    """An LDS-DMA load takes its LDS address from m0: between the scalar write of m0 and the load stands another
    instruction, in every GEMM kernel."""
    from triton_chip_benchmarks_amd import _native, audit

    seen = 0
    for name in _native.kernel_names():
        if not name.startswith("gemm_") or name.endswith("_checked"):
            continue
        body = audit.instructions(name)
        for before, line in zip(body, body[1:]):
            if line.split("//")[0].rstrip().endswith(" lds"):
                seen += 1
                destination = before.split(",")[0].split()[1:]
                assert destination != ["m0"], (name, before, line)
    assert seen > 1000
