"""The work this library is measured on: complex GEMM, transposes and packing through the public
classes (`Pipeline`, `GEMM`, `Transpose`, `Packing`), from one small product to the large batched
ones, on every input type.

A case is a dict of plain values:

    path      how the caller goes in:
                pipeline   Pipeline.Run on the caller's matrices (1-bit: one byte per sample)
                host       Pipeline.RunHost on page-locked host buffers
                basic      GEMM(Variant.basic).Run on planar matrices
                steps      [Packing ->] Transpose.RunPair -> GEMM(Variant.opt).Run
                packing    Packing forward, then backward
    B M N K   sizes (packing: N samples)
    tin tout  ValueType names
    axis_in axis_out  "planar" / "interleaved"
    order     "row" / "col": layout of C
    alpha, beta (real and imaginary parts)
"""
import math

import torch

import ccglib_amd as cc

VT, AX, MO = cc.ValueType, cc.ComplexAxisLocation, cc.MemOrder
AXIS = {"planar": AX.complex_planar, "interleaved": AX.complex_interleaved}
ORDER = {"row": MO.row_major, "col": MO.col_major}
TORCH = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32,
         "float8e4m3": torch.float8_e4m3fn, "float8e5m2": torch.float8_e5m2, "int32": torch.int32}
BYTES = {"float16": 2, "bfloat16": 2, "float32": 4, "float8e4m3": 1, "float8e5m2": 1, "int32": 4,
         "int1": 1}        # (the caller's 1-bit samples are one byte each)
F8_MAX = {"float8e4m3": 448.0, "float8e5m2": 57344.0}


def _case(path, B, M, N, K, tin, tout, axis_in="planar", axis_out="planar", order="row",
          alpha=(1.0, 0.0), beta=(0.0, 0.0), name=None):
    case = {"path": path, "B": B, "M": M, "N": N, "K": K, "tin": tin, "tout": tout,
            "axis_in": axis_in, "axis_out": axis_out, "order": order, "alpha_re": alpha[0],
            "alpha_im": alpha[1], "beta_re": beta[0], "beta_im": beta[1]}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # One small product, launch latency: the configuration the CPU reference is quoted on.
        _case("pipeline", 1, 256, 256, 256, "float16", "float32", name="cube256_f16"),
        # A handful of small matrices accumulated into C with complex factors, column-major, rows
        # one short of a tile: the shape of the library's alpha / beta tests.
        _case("basic", 16, 255, 128, 256, "bfloat16", "float32", order="col",
              alpha=(0.3, 1.6), beta=(0.5, -0.25), name="batch16_accumulate_bf16"),
        # One frequency channel of a beamformer handed over in host memory.
        _case("host", 1, 512, 1024, 576, "float16", "float32", axis_in="interleaved",
              name="channel_from_host_f16"),
        # Correlator of a small array: many channels, few receivers, samples as they arrive.
        _case("pipeline", 256, 96, 96, 1024, "float16", "float32", axis_in="interleaved",
              name="correlator96_f16"),
        # Beamformer with sizes that fit no tile, (re, im) pairs in and out.
        _case("pipeline", 16, 300, 3001, 577, "float16", "float32", axis_in="interleaved",
              axis_out="interleaved", name="beamformer_ragged_f16"),
        # 32-bit product of ordinary size, column-major result.
        _case("pipeline", 2, 1000, 1000, 1000, "float32", "float32", order="col",
              name="cube1000_f32"),
        # The beamformer of the benchmark through the one call that takes its raw samples ...
        _case("pipeline", 64, 512, 4096, 576, "float16", "float32", axis_in="interleaved",
              name="beamformer_f16"),
        # ... and step by step, as the benchmark does it by default.
        _case("steps", 64, 512, 4096, 576, "float16", "float32", axis_in="interleaved",
              name="beamformer_steps_f16"),
        # Bit packing and unpacking on their own, a sample count that ends inside a word.
        _case("packing", 1, 1, 1000000007, 1, "int1", "int32", name="pack_unpack"),
        # Large square product with 16-bit result.
        _case("pipeline", 1, 8192, 8192, 8192, "bfloat16", "bfloat16", name="cube8192_bf16"),
        # 8-bit batched product.
        _case("pipeline", 16, 4096, 4096, 8192, "float8e4m3", "float32", name="batch16_fp8"),
        # 1-bit correlator on raw samples.
        _case("pipeline", 32, 1024, 1024, 65536, "int1", "int32", name="correlator1024_int1"),
    ]


# Rates that keep a drawn case below the listed ones (ops/s), and the seconds it may take by them.
_RATE = {"float16": 1.2e15, "bfloat16": 1.2e15, "float32": 1.2e14, "float8e4m3": 2.4e15,
         "float8e5m2": 2.4e15, "int1": 5e15}
_MOST_S = 4e-3


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _extent(rng, low, high):
    """A size between low and high: as it falls, or rounded to a multiple that arrays often have."""
    n = _log(rng, low, high)
    step = rng.choice([1, 1, 8, 32, 64, 128])
    return max(low, min(high, (n + step // 2) // step * step))


def draw(rng):
    """One case of the ranges the listed ones stand for."""
    path = rng.choice(["pipeline", "pipeline", "pipeline", "basic", "steps", "host", "packing"])
    if path == "packing":
        return _case("packing", 1, 1, _log(rng, 1 << 16, 1 << 30), 1, "int1", "int32")
    one_bit = path in ("pipeline", "steps") and rng.random() < 0.2
    if one_bit:
        tin, tout = "int1", "int32"
    else:
        tin, tout = rng.choice([("float16", "float32"), ("float16", "float32"),
                                ("float16", "float16"), ("bfloat16", "float32"),
                                ("bfloat16", "bfloat16"), ("float32", "float32"),
                                ("float8e4m3", "float32"), ("float8e5m2", "float32")])
    axis_in = "planar" if path == "basic" else rng.choice(["planar", "interleaved"])
    axis_out = "planar" if path == "basic" else rng.choice(["planar", "planar", "interleaved"])
    order = rng.choice(["row", "row", "col"])
    alpha, beta = (1.0, 0.0), (0.0, 0.0)
    if not one_bit and rng.random() < 0.25:
        alpha = (round(rng.uniform(-2, 2), 2), round(rng.uniform(-2, 2), 2))
        if rng.random() < 0.5:   # (modulus below 1: C stays bounded however often a pass is repeated)
            beta = (round(rng.uniform(-0.6, 0.6), 2), round(rng.uniform(-0.6, 0.6), 2))
    if one_bit and path == "steps":
        axis_in = "planar"       # Packing has de-interleaved the bits by then
    while True:
        B = _log(rng, 1, 256)
        if one_bit:
            M, N, K = _extent(rng, 32, 1024), _extent(rng, 32, 1024), 32 * _log(rng, 16, 2048)
        else:
            M, N, K = _extent(rng, 16, 4096), _extent(rng, 32, 8192), _extent(rng, 32, 8192)
        case = _case(path, B, M, N, K, tin, tout, axis_in, axis_out, order, alpha, beta)
        w = work(case)
        if path == "host":
            if w["bytes"] <= 64e6:
                return case
        elif w["flops"] / _RATE[tin] <= _MOST_S and w["bytes"] <= 8e9:
            return case


def _matrix(case, rows, phases, gen):
    """The caller's matrix: unit phases (beam weights) or complex Gaussian samples; 1-bit samples
    are fair coins, one byte each."""
    B, K, tin = case["B"], case["K"], case["tin"]
    interleaved = case["axis_in"] == "interleaved"
    shape = (B, rows, K, 2) if interleaved else (B, 2, rows, K)
    if tin == "int1":
        return torch.randint(0, 2, shape, device="cuda", generator=gen, dtype=torch.uint8)
    if phases:
        angle = torch.rand((B, rows, K), device="cuda", generator=gen) * (2 * math.pi)
        x = torch.stack([torch.cos(angle), torch.sin(angle)], dim=3 if interleaved else 1)
    else:
        x = torch.randn(shape, device="cuda", generator=gen)
    if tin in F8_MAX:
        x = (x * (F8_MAX[tin] / x.abs().max())).clamp_(-F8_MAX[tin], F8_MAX[tin])
    return x.to(TORCH[tin]).contiguous()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    stream = torch.cuda.current_stream().cuda_stream
    path, B, M, N, K = case["path"], case["B"], case["M"], case["N"], case["K"]
    if path == "packing":
        samples = torch.randint(0, 2, (N,), device="cuda", generator=gen, dtype=torch.uint8)
        return {"path": path, "samples": samples,
                "words": torch.empty(cc.ceildiv(N, 32), dtype=torch.int32, device="cuda"),
                "back": torch.empty_like(samples),
                "pack": cc.Packing(N, cc.Direction.forward, 0, stream),
                "unpack": cc.Packing(N, cc.Direction.backward, 0, stream)}
    tin, tout = VT[case["tin"]], VT[case["tout"]]
    axis_in, axis_out, order = AXIS[case["axis_in"]], AXIS[case["axis_out"]], ORDER[case["order"]]
    alpha = complex(case["alpha_re"], case["alpha_im"])
    beta = complex(case["beta_re"], case["beta_im"])
    # (a beamformer's weights against its samples; a correlator has samples on both sides)
    a = _matrix(case, M, M != N, gen)
    b = _matrix(case, N, False, gen)
    rows, cols = (M, N) if case["order"] == "row" else (N, M)
    c_shape = (B, rows, cols, 2) if case["axis_out"] == "interleaved" else (B, 2, rows, cols)
    c = torch.zeros(c_shape, dtype=TORCH[case["tout"]], device="cuda")
    state = {"path": path, "a": a, "b": b, "c": c}
    if path in ("pipeline", "host"):
        state["pipeline"] = cc.Pipeline(B, M, N, K, 0, stream, axis_in, axis_out, MO.row_major,
                                        MO.col_major, order, tin, tout, cc.Variant.opt, alpha, beta)
        if path == "host":
            for k in ("a", "b", "c"):
                host = torch.empty(state[k].shape, dtype=state[k].dtype, pin_memory=True)
                state[k] = host.copy_(state[k])
        return state
    precision = cc.Precision(tin, tout)
    variant = cc.Variant.basic if path == "basic" else cc.Variant.opt
    state["gemm"] = cc.GEMM(B, M, N, K, 0, stream, precision, variant, axis_out, order,
                            MO.row_major, MO.col_major, alpha, beta)
    if path == "steps":
        bits = precision.GetInputBits()
        mb, nb, kc = cc.GEMM.GetDimensions(precision)
        k_padded = cc.ceildiv(K, kc) * kc
        for k, rows, chunk in (("a", M, mb), ("b", N, nb)):
            if tin == VT.int1:
                state["pack_" + k] = cc.Packing(B * 2 * rows * K, cc.Direction.forward, 0, stream)
                state["packed_" + k] = torch.empty(B * 2 * rows * K // 32, dtype=torch.int32,
                                                   device="cuda")
            state["transpose_" + k] = cc.Transpose(B, rows, K, chunk, kc, bits, 0, stream, axis_in)
            state["tiles_" + k] = torch.empty(
                B * 2 * cc.ceildiv(rows, chunk) * chunk * k_padded * bits // 8, dtype=torch.uint8,
                device="cuda")
    return state


def run(state):
    path = state["path"]
    if path == "packing":
        state["pack"].Run(state["samples"].data_ptr(), state["words"].data_ptr())
        state["unpack"].Run(state["words"].data_ptr(), state["back"].data_ptr())
        return {"words": state["words"], "back": state["back"]}
    a, b, c = state["a"], state["b"], state["c"]
    if path == "pipeline":
        state["pipeline"].Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
    elif path == "host":
        state["pipeline"].RunHost(a.data_ptr(), b.data_ptr(), c.data_ptr())
    elif path == "basic":
        state["gemm"].Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
    else:
        if "pack_a" in state:
            state["pack_a"].Run(a.data_ptr(), state["packed_a"].data_ptr())
            state["pack_b"].Run(b.data_ptr(), state["packed_b"].data_ptr())
            a, b = state["packed_a"], state["packed_b"]
        cc.Transpose.RunPair(state["transpose_a"], a.data_ptr(), state["tiles_a"].data_ptr(),
                             state["transpose_b"], b.data_ptr(), state["tiles_b"].data_ptr())
        state["gemm"].Run(state["tiles_a"].data_ptr(), state["tiles_b"].data_ptr(), c.data_ptr())
    return {"c": c}


def work(case):
    B, M, N, K = case["B"], case["M"], case["N"], case["K"]
    if case["path"] == "packing":
        return {"bytes": 2 * (N + cc.ceildiv(N, 32) * 4), "flops": 0}
    c_bytes = B * 2 * M * N * BYTES[case["tout"]]
    reads_c = case["beta_re"] != 0 or case["beta_im"] != 0
    return {"bytes": B * 2 * (M + N) * K * BYTES[case["tin"]] + c_bytes * (2 if reads_c else 1),
            "flops": 8 * B * M * N * K}


def tolerance(case):
    """Bits and whole numbers are exact. Floating-point results differ by the order of the fp32
    sums and, for a 16-bit C, by the rare element that then rounds to the other neighbour. About
    four times what separates the results from a product in 64 bits rounded to the type of C."""
    if case["tin"] == "int1":
        return "exact"
    if case["tout"] == "float16":      # measured: rel up to 2.4e-5; one step of the type 9.7e-4
        return {"rel": 1e-4, "max": 4e-3}
    if case["tout"] == "bfloat16":     # measured: rel up to 5.8e-5; one step of the type 7.8e-3
        return {"rel": 2.5e-4, "max": 3e-2}
    if case["tin"] in F8_MAX:          # measured: rel up to 1.5e-5, max 8.4e-5
        return {"rel": 6e-5, "max": 3.5e-4}
    return {"rel": 4e-6, "max": 3e-5}  # measured: rel up to 8.0e-7, max 6.2e-6


def exact(case, seed):
    """The product in 64 bits, one batch at a time (a fresh C is zero, so beta adds nothing); None
    where the outputs are bits."""
    if case["path"] == "packing":
        return None
    state = prepare(case, seed)
    planes = []
    for x in (state["a"].cuda(), state["b"].cuda()):
        x = x.movedim(3, 1) if case["axis_in"] == "interleaved" else x   # [B][2][rows][K]
        planes.append(x * 2.0 - 1.0 if case["tin"] == "int1" else x)     # (a 1-bit sample is +1 or -1)
    a, b = planes
    alpha = complex(case["alpha_re"], case["alpha_im"])
    c = torch.zeros(state["c"].shape, dtype=torch.float64, device="cuda")
    for i in range(case["B"]):
        (ar, ai), (br, bi) = a[i].double(), b[i].double()
        brt, bit = br.t().contiguous(), bi.t().contiguous()
        re, im = ar @ brt - ai @ bit, ar @ bit + ai @ brt
        re, im = alpha.real * re - alpha.imag * im, alpha.real * im + alpha.imag * re
        if case["order"] == "col":
            re, im = re.t(), im.t()
        c[i] = torch.stack([re, im], dim=2 if case["axis_out"] == "interleaved" else 0)
    return {"c": c}
