"""Where reading rows in place stops paying: Pipeline.Run with the GEMM reading the caller's
rows in place (option PIPELINE_ROUTE = 1) against the two transposes followed by the GEMM on
tiles (PIPELINE_ROUTE = 2), for shapes on either side of the break-even points that
ccglib_pipeline_create uses (M N / (M + N): what the GEMM's work grows with, over what the
transposes' grows with), and the route the default picks.

    python -m ccglib_amd.tuning.pipeline_crossover [--k 256] [--rounds 3]
    python -m ccglib_amd.tuning.pipeline_crossover --random 150 [--seed 1] [--input fp32] [--csv FILE]

One MI355X, synthetic operands (N(0, 1); fp8 scaled into range), device buffers; every
(shape, route) is warmed up and then timed over about 40 ms of back-to-back Runs between
two events, `rounds` times in alternation; the table holds the medians.

--random: that many problems of every family, rows that are whole 16-byte chunks and ragged ones, of
sizes spread over their logarithm (B to 256, M and N 16 to 8192, K from 16 bytes a row to 8192, up to about 2 ms and
2 GB of operands), every Run on other operands out of 512 MB of them, both routes in turn about 4 ms
at a time. For every family: the mean of log(time / time on tiled copies) of the default and of the better route,
and where the default is slower than the better one by more than 8 %.
"""
import argparse
import math
import random
import statistics

import torch

import ccglib_amd as cc

VT, AX, MO = cc.ValueType, cc.ComplexAxisLocation, cc.MemOrder
FAMILIES = [
    ("fp16 interleaved rows", VT.float16, torch.float16, AX.complex_interleaved),
    ("fp8 e4m3 interleaved rows", VT.float8e4m3, torch.float8_e4m3fn, AX.complex_interleaved),
    ("fp16 planar rows", VT.float16, torch.float16, AX.complex_planar),
]
# (M, N): squares across the break-even points, and rectangles to check that M N / (M + N) is
# the right abscissa
SHAPES = [(2048, 2048), (3072, 3072), (4096, 4096), (5120, 5120), (6144, 6144), (7168, 7168),
          (8192, 8192), (12288, 12288), (2048, 16384), (4096, 16384), (4096, 32768), (512, 4096)]


def time_runs(pipe, a, b, c, budget_ms=40.0):
    stream = torch.cuda.current_stream()
    for _ in range(3):
        pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
    e1.record(stream)
    e1.synchronize()
    n = max(3, int(budget_ms / max(e0.elapsed_time(e1), 1e-3)))
    e0.record(stream)
    for _ in range(n):
        pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
    e1.record(stream)
    e1.synchronize()
    return e0.elapsed_time(e1) / n


RANDOM_FAMILIES = [(name, vt, tdt, axis, ragged)
                   for name, vt, tdt, axis in FAMILIES + [
                       ("fp8 e4m3 planar rows", VT.float8e4m3, torch.float8_e4m3fn, AX.complex_planar),
                       ("fp32 interleaved rows", VT.float32, torch.float32, AX.complex_interleaved),
                       ("fp32 planar rows", VT.float32, torch.float32, AX.complex_planar)]
                   for ragged in (False, True)]
RATE = {VT.float16: 1.0e15, VT.float8e4m3: 2.0e15, VT.float32: 1.3e14}


def random_problem(rng, vt, axis, ragged):
    """B, M, N, K, C's axis."""
    size = {VT.float16: 2, VT.float8e4m3: 1, VT.float32: 4}[vt]
    chunk = 16 // size // (2 if axis == AX.complex_interleaved else 1)   # values of K in 16 bytes of a row

    def log(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    while True:
        B, M, N, K = log(1, 256), log(16, 8192), log(16, 8192), log(chunk, 8192)
        step = rng.choice([1, 16, 64])
        M, N = max(16, M // step * step), max(16, N // step * step)
        K = K // chunk * chunk
        if ragged:
            if chunk == 1:
                continue
            K += rng.randrange(1, chunk)
        if 8 * B * M * N * K / RATE[vt] <= 2e-3 and B * 2 * (M + N) * K * size <= 2e9 and B * M * N <= 2.5e8:
            return B, M, N, K, rng.choice([AX.complex_planar, AX.complex_planar, AX.complex_interleaved])


def random_problems(args, s):
    rng = random.Random(args.seed)
    gen = torch.Generator(device="cuda").manual_seed(1)
    csv = open(args.csv, "w") if args.csv else None
    print("%-34s %8s   %10s %10s   %s" % ("family", "problems", "default", "better", "default > 8 % slower, at worst"))
    for name, vt, tdt, axis, ragged in RANDOM_FAMILIES:
        if args.input and not name.startswith(args.input):
            continue
        scale = 448.0 / 5.8 if vt == VT.float8e4m3 else 1.0
        noise = (torch.randn(1 << 28, device="cuda", generator=gen) * scale).to(tdt)   # (from 256 MB on)
        size = noise.element_size()
        results = []
        for _ in range(args.random):
            B, M, N, K, c_axis = random_problem(rng, vt, axis, ragged)
            pipes = {}
            for route in (0, 1, 2):
                with cc.option(cc.Option.pipeline_route, route):
                    pipes[route] = cc.Pipeline(B, M, N, K, 0, s, axis, c_axis, MO.row_major, MO.col_major,
                                               MO.row_major, vt, VT.float32, cc.Variant.opt)
            assert pipes[1].ReadsInPlace() and not pipes[2].ReadsInPlace()
            step_a, step_b = ((B * 2 * rows * K * size + 255) // 256 * 256 for rows in (M, N))
            slots = max(1, min(256, (1 << 29) // (step_a + step_b)))
            a = noise[:0].new_empty(slots * step_a // size)
            b = noise[:0].new_empty(slots * step_b // size)
            for x in (a, b):
                for at in range(0, x.numel(), noise.numel()):
                    x[at:at + noise.numel()] = noise[:min(noise.numel(), x.numel() - at)]
            c = torch.empty(B * 2 * M * N, device="cuda")
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            at = 0

            def runs(pipe, n):
                nonlocal at
                for _ in range(n):
                    at = (at + 1) % slots
                    pipe.Run(a.data_ptr() + at * step_a, b.data_ptr() + at * step_b, c.data_ptr())

            def once(pipe, n):
                e0.record()
                runs(pipe, n)
                e1.record()
                e1.synchronize()
                return e0.elapsed_time(e1) / n

            n = {}
            for route in (1, 2):
                runs(pipes[route], 2)
                n[route] = max(2, min(200, int(4.0 / once(pipes[route], 3))))
            times = {1: [], 2: []}
            for _ in range(args.rounds):
                for route in (1, 2):
                    times[route].append(once(pipes[route], n[route]))
            t1, t2 = statistics.median(times[1]), statistics.median(times[2])
            in_place = pipes[0].ReadsInPlace()
            results.append((t1, t2, in_place))
            if csv:
                csv.write("%s,%d,%d,%d,%d,%d,%d,%.5f,%.5f,%d\n" % (name, ragged, c_axis, B, M, N, K, t1, t2, in_place))
                csv.flush()
            del pipes, a, b, c
        chosen = [t1 if i else t2 for t1, t2, i in results]
        best = [min(t1, t2) for t1, t2, _ in results]
        behind = [x / y for x, y in zip(chosen, best)]
        mean = [math.exp(statistics.mean(math.log(x / t2) for x, (_, t2, _) in zip(v, results))) for v in (chosen, best)]
        print("%-34s %8d   %10.3f %10.3f   %.1f %%, %.2f" % (
            name + (", ragged" if ragged else ""), len(results), mean[0], mean[1],
            100.0 * sum(x > 1.08 for x in behind) / len(behind), max(behind)), flush=True)
        del noise


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--k", type=int, default=256)
    ap.add_argument("--rounds", type=int, default=3)
    ap.add_argument("--random", type=int, default=0)
    ap.add_argument("--seed", type=int, default=1)
    ap.add_argument("--input", help="only families whose name begins like this")
    ap.add_argument("--csv")
    args = ap.parse_args()
    if args.random:
        return random_problems(args, torch.cuda.current_stream().cuda_stream)
    K = args.k
    s = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(1)
    print("Pipeline.Run, opt variant, planar fp32 C, K = %d; B fills the compute units" % K)
    for name, vt, tdt, axis in FAMILIES:
        print("\n%s" % name)
        print("%-16s %4s %10s   %12s %12s   %8s   %s" % ("M x N", "B", "MN/(M+N)", "in place ms", "transposed ms",
                                                       "ratio", "default route"))
        for M, N in SHAPES:
            B = max(1, (1 << 27) // (M * N))
            shape_a = (B, M, K, 2) if axis == AX.complex_interleaved else (B, 2, M, K)
            shape_b = (B, N, K, 2) if axis == AX.complex_interleaved else (B, 2, N, K)
            scale = 448.0 / 5.8 if vt == VT.float8e4m3 else 1.0
            a = (torch.randn(shape_a, device="cuda", generator=gen) * scale).to(tdt)
            b = (torch.randn(shape_b, device="cuda", generator=gen) * scale).to(tdt)
            c = torch.empty((B, 2, M, N), device="cuda")
            pipes = {}
            for route in (0, 1, 2):
                with cc.option(cc.Option.pipeline_route, route):
                    pipes[route] = cc.Pipeline(B, M, N, K, 0, s, axis, AX.complex_planar, MO.row_major,
                                               MO.col_major, MO.row_major, vt, VT.float32, cc.Variant.opt)
            assert pipes[1].ReadsInPlace() and not pipes[2].ReadsInPlace()
            times = {1: [], 2: []}
            for _ in range(args.rounds):
                for route in (1, 2):
                    times[route].append(time_runs(pipes[route], a, b, c))
            t1, t2 = statistics.median(times[1]), statistics.median(times[2])
            print("%-16s %4d %10.0f   %12.4f %12.4f   %8.3f   %s" % (
                "%d x %d" % (M, N), B, M * N / (M + N), t1, t2, t1 / t2,
                "in place" if pipes[0].ReadsInPlace() else "transposed"), flush=True)
            del pipes, a, b, c


if __name__ == "__main__":
    main()
