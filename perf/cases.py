"""The calls whose speed a user of this suite sees, measured one pass at a time.

Each case is one launch of a public entry point as the benchmark programs make
it: an HBM copy or read (bench_bandwidth), a vector chain (bench_vector), a
resident matrix tile (bench_tensor, peak mode) or a GEMM (bench_tensor, gemm
mode), over the sizes, types, tiles and options those programs accept.
`listed` names the ones compared from change to change; `draw` spreads more
over the same ranges.
"""

from __future__ import annotations

import math

import torch

from triton_chip_benchmarks_amd import _native, bench_bandwidth, bench_tensor, bench_vector, formats

DEVICE = "cuda"
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16, "fp64": torch.float64,
          "int8": torch.int8, "fp8": torch.float8_e4m3fn}
ELEM_BITS = {"bf16": 16, "fp16": 16, "fp32": 32, "fp64": 64, "int8": 8, "fp8": 8, "fp4": 4}
# Dense matrix rates relative to BF16, to bound a drawn case's time by the largest listed one's.
MATRIX_RATE = {"bf16": 1.0, "fp16": 1.0, "int8": 2.0, "fp8": 2.0, "fp4": 4.0, "fp32": 1 / 16, "fp64": 1 / 32}
VECTOR_STORE = {"fp32": torch.float32, "fp64": torch.float64, "fp16": torch.float16, "bf16_dot2": torch.bfloat16,
                "int8": torch.int32}
CHAINS = 8


def _gemm(name, dtype, m, n, k, tile="largest"):
    return {"name": name, "op": "gemm", "dtype": dtype, "m": m, "n": n, "k": k, "tile": tile}


def listed():
    return [
        # The copy program's smoke buffer (8 MiB of fp32) with a ragged end: launch latency and the cache regime.
        {"name": "copy_fp32_8mib_ragged", "op": "copy", "dtype": "fp32", "elements": (1 << 21) + 17, "offset": 0,
         "threads": 256, "vectors": 1, "policy": "off"},
        # The headline copy: 2^28 fp32, one wave per workgroup, streaming policy.
        {"name": "copy_fp32_1gib", "op": "copy", "dtype": "fp32", "elements": 1 << 28, "offset": 0, "threads": 64,
         "vectors": 1, "policy": "stream"},
        # The read sweep's smallest buffer and block: one sum per 256 values of a 256 MiB bf16 buffer.
        {"name": "read_bf16_256mib_block256", "op": "read", "dtype": "bf16", "elements": 1 << 27, "block": 256,
         "threads": 256},
        # The vector sweep's default launch: 8 workgroups of 256 lanes per CU, 4096 FMA updates.
        {"name": "vector_fp32", "op": "vector", "kind": "fp32", "elements": 8 * 256 * 256, "iterations": 4096,
         "unroll": 8, "threads": 256},
        # A resident BF16 tile, two chains, the peak sweep's 4 workgroups per CU and 1024 repeats.
        {"name": "peak_bf16_128x128x64", "op": "peak", "dtype": "bf16", "tile_m": 128, "chains": 2, "blocks": 1024,
         "iterations": 1024},
        # The GEMM program's smoke size: one launch is all latency.
        _gemm("gemm_bf16_256", "bf16", 256, 256, 256),
        # A ragged shape off every tile on the smallest tile of the sweep, as the reference-recipe check runs it.
        _gemm("gemm_fp16_1000x744x1000", "fp16", 1000, 744, 1000, "smallest"),
        # The reference recipe's sizes start at 2048: fewer large tiles than CUs.
        _gemm("gemm_bf16_2048", "bf16", 2048, 2048, 2048),
        _gemm("gemm_fp64_2048", "fp64", 2048, 2048, 2048),
        # A layer-sized FP8 product whose M, N and K fit no tile.
        _gemm("gemm_fp8_5000x3000x4112", "fp8", 5000, 3000, 4112),
        # MXFP4 at an ordinary square size, block scales of a spread of magnitudes.
        _gemm("gemm_fp4_4096", "fp4", 4096, 4096, 4096),
        # The headline BF16 GEMM.
        _gemm("gemm_bf16_8192", "bf16", 8192, 8192, 8192),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_gemm(rng):
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp8", "fp8", "fp4", "int8", "fp32", "fp64"])
    most = 8192.0**3 * MATRIX_RATE[dtype]
    row = 128 // ELEM_BITS[dtype]  # elements per 16-byte row unit
    while True:
        if rng.random() < 0.4:  # square, as the program's --sizes
            m = n = k = 64 * _log_uniform(rng, 2, 128)
        else:
            m, n, k = (_log_uniform(rng, 64, 8192) for _ in range(3))
            if rng.random() < 0.3:
                m, n, k = (-(-x // 128) * 128 for x in (m, n, k))
        k = -(-k // row) * row
        if m * n * k <= most:
            return {"op": "gemm", "dtype": dtype, "m": m, "n": n, "k": k,
                    "tile": rng.choice(["largest", "largest", "smallest"])}


def draw(rng):
    pick = rng.random()
    if pick < 0.6:
        return _draw_gemm(rng)
    if pick < 0.75:
        # Tensors of any length; a slice of a tensor starts off the 16-byte grid.
        return {"op": "copy", "dtype": rng.choice(["fp32", "fp16", "bf16"]),
                "elements": _log_uniform(rng, 1 << 10, 1 << 28), "offset": rng.choice([0, 0, 0, 1]),
                "threads": rng.choice([64, 256, 512]), "vectors": rng.choice([1, 2, 4]),
                "policy": rng.choice(["off", "on", "stream"])}
    if pick < 0.88:
        return {"op": "read", "dtype": rng.choice(["fp32", "fp16", "bf16"]),
                "elements": _log_uniform(rng, 1 << 14, 1 << 28), "block": rng.choice([256, 1024, 4096, 16384]),
                "threads": rng.choice([64, 256, 512])}
    if pick < 0.95:
        threads = rng.choice([256, 512, 1024])
        return {"op": "vector", "kind": rng.choice(["fp32", "fp16", "bf16_dot2", "fp64", "int8"]),
                "elements": threads * rng.randint(64, 4096 * 256 // threads), "iterations": 4096 // 2**rng.randint(2, 6),
                "unroll": rng.choice([4, 8, 16]), "threads": threads}
    return {"op": "peak", "dtype": rng.choice(["bf16", "fp16", "int8", "fp8"]), "tile_m": rng.choice([64, 128, 256]),
            "chains": 0, "blocks": rng.randint(64, 1024), "iterations": 2**rng.randint(5, 9)}


# ---- operands ----------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _random_scales(rows, k, generator):
    """E8M0 codes of one scale per 32 K elements, 2^-3 .. 2^3, row-major [rows][ceil(K/32)]."""
    return torch.randint(124, 131, (rows, k // formats.MX_GROUP_SIZE), device=DEVICE, generator=generator,
                         dtype=torch.uint8)


def _gemm_operands(case, seed):
    """(a, b, row-major scales or None): B stored [n][k]; N(0,1) A and N(0,1)/sqrt(K) B rounded to the format
    (FP8 both N(0,1)), INT8 over its whole range, MXFP4 codes over all sixteen values."""
    dtype, m, n, k = case["dtype"], case["m"], case["n"], case["k"]
    generator = _generator(seed)
    if dtype == "fp4":
        codes = [torch.randint(0, 16, (rows, k), device=DEVICE, generator=generator, dtype=torch.uint8)
                 for rows in (m, n)]
        return codes[0], codes[1], tuple(_random_scales(rows, k, generator) for rows in (m, n))
    if dtype == "int8":
        return tuple(torch.randint(-128, 128, (rows, k), device=DEVICE, generator=generator, dtype=torch.int8)
                     for rows in (m, n)) + (None,)
    drawn = torch.float64 if dtype == "fp64" else torch.float32
    a = torch.randn((m, k), device=DEVICE, generator=generator, dtype=drawn)
    b = torch.randn((n, k), device=DEVICE, generator=generator, dtype=drawn)
    if dtype != "fp8":
        b *= 1.0 / math.sqrt(k)
    return a.to(DTYPES[dtype]), b.to(DTYPES[dtype]), None


def _gemm_tile(case):
    configs = _native.gemm_configs(case["dtype"])
    return (max if case["tile"] == "largest" else min)(configs, key=lambda c: c["tile_m"] * c["tile_n"])


def _peak_config(case):
    return next(c for c in _native.peak_configs(case["dtype"])
                if c["tile_m"] == case["tile_m"] and not c["b_nk"] and c["mfma_m"] == 32
                and case["chains"] in (0, c["chains"]))


def _uniform(elements, dtype, generator):
    return torch.empty(elements, device=DEVICE, dtype=DTYPES[dtype]).uniform_(-1, 1, generator=generator)


def _vector_operands(case, seed):
    """States x0 ~ U[0.5, 1), a = 0.999, b = 1e-3; INT8: state words with bytes of [-4, 4], weights and bias 1."""
    kind, elements = case["kind"], case["elements"]
    generator = _generator(seed)
    if kind == "int8":
        inputs = torch.randint(-4, 5, (CHAINS, elements), device=DEVICE, generator=generator, dtype=torch.int32)
        return inputs, torch.tensor([0x01010101] + [1] * CHAINS, dtype=torch.int32, device=DEVICE)
    drawn = torch.float64 if kind == "fp64" else torch.float32
    inputs = torch.empty((CHAINS, elements), device=DEVICE, dtype=drawn).uniform_(0.5, 1.0, generator=generator)
    store = VECTOR_STORE[kind]
    return inputs.to(store), torch.tensor([0.999] + [1e-3] * CHAINS, dtype=torch.float64).to(store).to(DEVICE)


def prepare(case, seed):
    op = case["op"]
    if op == "copy":
        offset = case["offset"]
        src = _uniform(case["elements"] + offset, case["dtype"], _generator(seed))
        return {"case": case, "src": src[offset:], "dst": torch.empty_like(src)[offset:]}
    if op == "read":
        src = _uniform(case["elements"], case["dtype"], _generator(seed))
        return {"case": case, "src": src,
                "sink": torch.empty(-(-case["elements"] // case["block"]), device=DEVICE)}
    if op == "vector":
        inputs, coefficients = _vector_operands(case, seed)
        if case["kind"] == "bf16_dot2":  # once per operand set, as the program does before it times launches
            bench_vector.require_dot2_regime(inputs, coefficients, case["iterations"])
        return {"case": case, "inputs": inputs, "coefficients": coefficients, "output": torch.empty_like(inputs)}
    if op == "peak":
        config = _peak_config(case)
        a, b, c, _ = bench_tensor.peak_inputs(case["blocks"], config, case["dtype"], DEVICE, seed)
        return {"case": case, "config": config, "a": a, "b": b, "c": c}
    a, b, scales = _gemm_operands(case, seed)
    if case["dtype"] == "fp4":
        a, b = formats.pack_e2m1_pairs(a), formats.pack_e2m1_pairs(b)
        scales = tuple(formats.mx_scale_blocks(s) for s in scales)
    out = {"int8": torch.int32, "fp64": torch.float64}.get(case["dtype"], torch.float32)
    return {"case": case, "config": _gemm_tile(case), "a": a, "b": b, "scales": scales or (None, None),
            "c": torch.empty((case["m"], case["n"]), dtype=out, device=DEVICE)}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "copy":
        bench_bandwidth.launch_copy(state["src"], state["dst"], case["threads"], case["vectors"], 0, case["policy"])
        return state["dst"]
    if op == "read":
        bench_bandwidth.launch_read(state["src"], state["sink"], case["block"], case["threads"])
        return state["sink"]
    if op == "vector":
        bench_vector.launch_vector(case["kind"], state["inputs"], state["output"], state["coefficients"],
                                   case["iterations"], case["unroll"], case["threads"], regime_checked=True)
        return state["output"]
    if op == "peak":
        bench_tensor.launch_peak(case["dtype"], state["config"], state["a"], state["b"], state["c"],
                                 case["iterations"])
        return state["c"]
    _native.gemm(case["dtype"], state["config"], state["a"], state["b"], state["c"], case["m"], case["n"], case["k"],
                 *state["scales"])
    return state["c"]


# ---- what a pass needs, and what it should give ----------------------------------


def work(case):
    op = case["op"]
    if op == "copy":
        return {"bytes": 2 * case["elements"] * DTYPES[case["dtype"]].itemsize, "flops": 0}
    if op == "read":
        return {"bytes": case["elements"] * DTYPES[case["dtype"]].itemsize + -(-case["elements"] // case["block"]) * 4,
                "flops": case["elements"]}
    if op == "vector":
        states = CHAINS * case["elements"]
        per_update = 8 if case["kind"] == "int8" else 2
        return {"bytes": 2 * states * VECTOR_STORE[case["kind"]].itemsize,
                "flops": per_update * states * case["iterations"]}
    if op == "peak":
        c = _peak_config(case)
        m, n, k, chains, blocks = c["tile_m"], c["tile_n"], c["tile_k"], c["chains"], case["blocks"]
        return {"bytes": blocks * ((m + chains * n) * k * ELEM_BITS[case["dtype"]] // 8 + chains * m * n * 4),
                "flops": 2 * m * n * k * chains * blocks * case["iterations"]}
    dtype, m, n, k = case["dtype"], case["m"], case["n"], case["k"]
    scales = (m + n) * (k // formats.MX_GROUP_SIZE) if dtype == "fp4" else 0
    return {"bytes": (m + n) * k * ELEM_BITS[dtype] // 8 + scales + m * n * (8 if dtype == "fp64" else 4),
            "flops": 2 * m * n * k}


def tolerance(case):
    op, dtype = case["op"], case.get("dtype")
    if op in ("copy", "peak") or dtype == "int8" or case.get("kind") in ("int8", "fp16", "bf16_dot2"):
        # Bytes, whole numbers, exact lattices, and chains whose every step rounds once to 16 bits.
        return "exact"
    # About four times the distance from the 64-bit result that the kernels showed at the largest sizes.
    if op == "vector":
        return {"rel": 1e-14 if case["kind"] == "fp64" else 4.5e-6}
    if op == "read":
        return {"rel": 1e-6}
    # The FP8 instructions drop low product bits inside one reduction: 1.3e-5 at every K, more than the sums add.
    return {"rel": {"fp64": 1e-14, "fp8": 6e-5}.get(dtype, 2.5e-6)}


def exact(case, seed):
    op = case["op"]
    if op == "copy":
        return _uniform(case["elements"] + case["offset"], case["dtype"], _generator(seed))[case["offset"]:].double()
    if op == "read":
        block = case["block"]
        values = _uniform(case["elements"], case["dtype"], _generator(seed)).double()
        padded = torch.nn.functional.pad(values, (0, -case["elements"] % block))
        return padded.view(-1, block).sum(dim=1)
    if op == "vector":
        if case["kind"] not in ("fp32", "fp64"):
            return None  # whole numbers, or a value that the 16-bit rounding of every step decides
        inputs, coefficients = _vector_operands(case, seed)
        coefficients = coefficients.double().cpu()
        a, b = coefficients[0].item(), coefficients[1:, None].to(DEVICE)
        decay = math.exp(case["iterations"] * math.log(a))
        return decay * inputs.double() + b * ((1.0 - decay) / (1.0 - a))
    if op == "peak":
        config = _peak_config(case)
        a, _, _, b = bench_tensor.peak_inputs(case["blocks"], config, case["dtype"], DEVICE, seed)
        a = a.double()
        return torch.stack([torch.matmul(a, chain.double().contiguous()) for chain in b]) * case["iterations"]
    a, b, scales = _gemm_operands(case, seed)
    if case["dtype"] == "fp4":
        a, b = (formats.e2m1_decode(codes) * formats.e8m0_decode(s).repeat_interleave(formats.MX_GROUP_SIZE, dim=1)
                for codes, s in zip((a, b), scales))
    return torch.matmul(a.double(), b.double().t().contiguous())
