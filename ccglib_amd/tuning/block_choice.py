"""How well the dispatch picks a block shape: GEMMs of random sizes, types, operand layouts and C
layouts, timed with each shape forced (option GEMM_BLOCK_TILE = 1, 2, 4: 256 x 128, 128 x 128,
64 x 64; 32-bit input has no 256 x 128; 5, 6, 7: waves of their own, where there are at most 2048 blocks of 64 x 64), and how far the
default is behind the fastest. One table for the problems whose default is a block (whichever forced shape the default's time is
closest to), against the three block shapes; one for those on waves, against 64 x 64 blocks and all shapes. The
constants of block_choice and wave_choice (../csrc/gemm_mfma.hip) are fitted to such times.

    python -m ccglib_amd.tuning.block_choice [--problems 2000] [--seed 1] [--warm] [--csv FILE] [--input float32]

One MI355X, N(0, 1) operands (fp8 scaled into range, random bits for 1-bit input). Every pass takes
other buffers, out of pools larger than the last-level cache; with --warm the same ones. The
shapes take turns, five times about 2 ms each; the medians count. Sizes: B up to 256, M and N 16 to
4096, K 64 to 4096 (1-bit: 512 to 32768), half of them multiples of 8 to 128, up to about 1.5 ms
and 1536 tiles of 256 x 128. K is a multiple of 16 (1-bit: 128); a third of the problems on rows in place
have any K ("ragged").
"""
import argparse
import collections
import math
import random
import statistics
import sys

import torch

import ccglib_amd as cc

VT, AX, MO = cc.ValueType, cc.ComplexAxisLocation, cc.MemOrder
SHAPES = {1: "256x128", 2: "128x128", 4: "64x64"}
PAIRS = [(VT.float16, VT.float32), (VT.float16, VT.float16), (VT.bfloat16, VT.bfloat16),
         (VT.float32, VT.float32), (VT.float32, VT.float16), (VT.float8e4m3, VT.float32),
         (VT.int1, VT.int32)]
BITS = {VT.float16: 16, VT.bfloat16: 16, VT.float32: 32, VT.float8e4m3: 8, VT.int1: 1, VT.int32: 32}
TORCH = {VT.float16: torch.float16, VT.bfloat16: torch.bfloat16, VT.float32: torch.float32,
         VT.float8e4m3: torch.float8_e4m3fn}
# operations per second that keep a problem below about 1.5 ms
RATE = {VT.float16: 1e15, VT.bfloat16: 1e15, VT.float32: 1.1e14, VT.float8e4m3: 2e15, VT.int1: 5e15}
POOL_BYTES = 1 << 31        # of each operand and of C
FOOTPRINT = 640e6           # what passes over other buffers touch before they come round


def log_size(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def extent(rng):
    n, step = log_size(rng, 16, 4096), rng.choice([1, 1, 8, 32, 64, 128])
    return max(16, (n + step // 2) // step * step)


def problem(rng, pairs):
    """(tin, tout, layout, C axis, alpha, beta, B, M, N, K) and the bytes of A, B and C."""
    while True:
        tin, tout = rng.choice(pairs)
        layout = rng.choice(["tiled", "tiled", "planar", "interleaved"])
        if layout == "interleaved" and tin == VT.int1:
            layout = "tiled"
        if layout != "tiled" and tin != VT.int1 and rng.random() < 0.33:
            layout += " ragged"
        c_axis = AX.complex_planar
        if not layout.startswith("planar") and rng.random() < 0.4:
            c_axis = AX.complex_interleaved
        alpha = 1 if rng.random() < 0.8 or tin == VT.int1 else 0.5 - 1.5j
        beta = 0 if rng.random() < 0.8 or tin == VT.int1 else 0.25 + 0.5j
        B, M, N = log_size(rng, 1, 256), extent(rng), extent(rng)
        K = (128 if tin == VT.int1 else 16) * log_size(rng, 4, 256)
        if layout.endswith("ragged"):
            K -= rng.randrange(1, 16)
        sizes = bytes_of(tin, tout, layout, B, M, N, K)
        if (8 * B * M * N * K / RATE[tin] <= 1.5e-3 and max(sizes) <= POOL_BYTES and
                B * cc.ceildiv(M, 128) * cc.ceildiv(N, 256) <= 1536):
            return (tin, tout, layout, c_axis, alpha, beta, B, M, N, K), sizes


def bytes_of(tin, tout, layout, B, M, N, K):
    """Bytes of A, B and C as the GEMM reads and writes them."""
    rows, k = [M, N], K
    if layout == "tiled":
        mb, nb, kc = cc.GEMM.GetDimensions(cc.Precision(tin, tout))
        rows, k = [cc.ceildiv(M, mb) * mb, cc.ceildiv(N, nb) * nb], cc.ceildiv(K, kc) * kc
    return [B * 2 * r * k * BITS[tin] // 8 for r in rows] + [B * 2 * M * N * BITS[tout] // 8]


# the problems that the comment of block_choice quotes
NAMED = [(VT.float16, VT.float32, "tiled", 0, 1, 4096, 4096, 512),
         (VT.float16, VT.float32, "tiled", 0, 5, 1024, 1024, 1024),
         (VT.float16, VT.float32, "tiled", 0, 256, 96, 96, 1024),
         (VT.float16, VT.float32, "tiled", 0, 1, 256, 256, 256),
         (VT.float16, VT.float16, "planar", 0, 167, 800, 184, 2064),
         (VT.float16, VT.float32, "planar", 0, 157, 192, 604, 3680),
         (VT.float32, VT.float32, "tiled", 0, 1, 4096, 4096, 512),
         (VT.float32, VT.float32, "tiled", 0, 2, 1000, 1000, 1000),
         (VT.float32, VT.float32, "interleaved", 0, 2, 1000, 1000, 1000),
         (VT.float8e4m3, VT.float32, "tiled", 0, 1, 4096, 4096, 512),
         (VT.float8e4m3, VT.float32, "tiled", 0, 1, 1024, 1024, 1024),
         (VT.float8e4m3, VT.float32, "planar", 0.25 + 0.5j, 11, 456, 1542, 192),
         (VT.int1, VT.int32, "tiled", 0, 1, 3452, 1504, 32256),
         (VT.int1, VT.int32, "tiled", 0, 1, 64, 64, 65536)]


_pools = {}


def pool(tin, which):
    key = (tin, which)
    if key not in _pools:
        if which == "c":
            x = torch.zeros(POOL_BYTES // 4, device="cuda")
        elif tin == VT.int1:
            x = torch.randint(-2 ** 31, 2 ** 31 - 1, (POOL_BYTES // 4,), dtype=torch.int32, device="cuda")
        elif tin == VT.float8e4m3:
            x = torch.cat([(torch.randn(POOL_BYTES // 8, device="cuda") * (448.0 / 5.8)).to(TORCH[tin])
                           for _ in range(8)])
        else:
            x = torch.randn(POOL_BYTES * 8 // BITS[tin], device="cuda", dtype=TORCH[tin])
        _pools[key] = x
    return _pools[key].data_ptr()


def make(case, block_tile):
    tin, tout, layout, c_axis, alpha, beta, B, M, N, K = case
    s = torch.cuda.current_stream().cuda_stream
    variant = cc.Variant.basic if layout.startswith("planar") else cc.Variant.opt
    with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, 1), \
            cc.option(cc.Option.basic_retile, 0):
        if layout.startswith("interleaved"):
            pipe = cc.Pipeline(B, M, N, K, 0, s, AX.complex_interleaved, c_axis, MO.row_major, MO.col_major,
                               MO.row_major, tin, tout, variant, alpha, beta)
            assert pipe.ReadsInPlace()
            return pipe
        return cc.GEMM(B, M, N, K, 0, s, cc.Precision(tin, tout), variant, c_axis, alpha=alpha, beta=beta)


def measure(case, sizes, warm):
    """Median microseconds of each shape and of the default."""
    steps = [(v + 511) // 512 * 512 for v in sizes]
    slots = 1 if warm else int(max(1, min(4096, FOOTPRINT // sum(steps), *(POOL_BYTES // v for v in steps))))
    base = [pool(case[0], "a"), pool(case[0], "b"), pool(None, "c")]
    where = [[p + i * v for p, v in zip(base, steps)] for i in range(slots)]
    tiles = [0, 2, 4] if case[0] == VT.float32 else [0, 1, 2, 4]
    if case[0] != VT.float32 and case[6] * cc.ceildiv(case[7], 64) * cc.ceildiv(case[8], 64) <= 2048:
        tiles += [5, 6, 7] if BITS[case[0]] == 16 else [5]
    runs = {t: make(case, t) for t in tiles}
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    at = 0

    def once(run, n):
        nonlocal at
        e0.record()
        for _ in range(n):
            at = (at + 1) % slots
            run.Run(*where[at])
        e1.record()
        e1.synchronize()
        return e0.elapsed_time(e1) / n * 1e3

    for r in runs.values():
        once(r, 3)
    n = max(4, min(200, int(2000 / once(runs[0], 5))))
    times = {t: [] for t in runs}
    for i in range(5):
        for t in (list(runs) if i % 2 else reversed(list(runs))):
            times[t].append(once(runs[t], n))
    medians = {t: statistics.median(v) for t, v in times.items()}
    medians.setdefault(1, math.nan)
    return medians


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--problems", type=int, default=2000)
    ap.add_argument("--seed", type=int, default=1)
    ap.add_argument("--warm", action="store_true")
    ap.add_argument("--csv")
    ap.add_argument("--input", help="only problems of this input type")
    args = ap.parse_args()
    pairs = [p for p in PAIRS if args.input in (None, p[0].name)]
    print("us: 256x128, 128x128, 64x64 on cold operands; on warm ones; default (warm)")
    for tin, tout, layout, beta, B, M, N, K in NAMED:
        if args.input not in (None, tin.name):
            continue
        case = (tin, tout, layout, AX.complex_planar, 1, beta, B, M, N, K)
        cold, warm = (measure(case, bytes_of(tin, tout, layout, B, M, N, K), w) for w in (False, True))
        print("%-52s %8.1f %8.1f %8.1f   %8.1f %8.1f %8.1f   %8.1f" % (
            "%s->%s %s%s B=%d %dx%dx%d" % (tin.name, tout.name, layout, " beta" if beta else "", B, M, N, K),
            cold[1], cold[2], cold[4], warm[1], warm[2], warm[4], warm[0]), flush=True)
    rng = random.Random(args.seed)
    groups, worst = collections.defaultdict(list), []
    csv = open(args.csv, "w") if args.csv else None
    for i in range(args.problems):
        case, sizes = problem(rng, pairs)
        t = measure(case, sizes, args.warm)
        tin, tout, layout, c_axis, alpha, beta, B, M, N, K = case
        text = "%s->%s %s%s%s B=%d %dx%dx%d" % (tin.name, tout.name, layout,
                                                " interleaved C" if c_axis == AX.complex_interleaved else "",
                                                " beta" if beta else "", B, M, N, K)
        times = {k: v for k, v in t.items() if k and v == v}
        waves = min(times, key=lambda k: abs(times[k] - t[0])) >= 5
        behind = t[0] / min(v for k, v in times.items() if waves or k < 5)
        for name in ("all", "%-12s %s" % (tin.name, layout)):
            groups[waves, name].append((behind, times[4] / t[0]))
        worst.append((behind, text, t))
        if csv:
            csv.write("%s,%s\n" % (text, ",".join("%d:%.2f" % kv for kv in sorted(t.items()))))
        if i % 200 == 199:
            print("%d problems" % (i + 1), file=sys.stderr, flush=True)
    for waves in (False, True):
        print("\n%s operands, default on %s" % (
            "warm" if args.warm else "cold",
            "waves: behind the fastest of blocks and waves, and 64x64 blocks over the default" if waves else
            "blocks: behind the fastest of 256x128, 128x128, 64x64 (192x256 blocks are then in front)"))
        print("%-30s %8s %14s %10s %10s%s" % ("input, layout", "problems", "mean behind %", "> 8 % in", "> 20 % in",
                                             "  64x64 / default" if waves else ""))
        for name in sorted(n for w, n in groups if w == waves):
            v = [x for x, _ in groups[waves, name]]
            over = [x for _, x in groups[waves, name]]
            print("%-30s %8d %14.2f %10d %10d%s" % (name, len(v), 100 * (statistics.mean(v) - 1),
                                                   sum(x > 1.08 for x in v), sum(x > 1.2 for x in v),
                                                   "%17.2f" % statistics.geometric_mean(over) if waves else ""))
    print("\nfarthest behind (us: default; 256x128, 128x128, 64x64; waves of 32x32, 32x16, 16x16)")
    for behind, text, t in sorted(worst, key=lambda w: -w[0])[:12]:
        print("%5.2f  %-66s %s" % (behind, text, " ".join("%8.1f" % t.get(k, math.nan) for k in (0, 1, 2, 4, 5, 6, 7))))


if __name__ == "__main__":
    main()
