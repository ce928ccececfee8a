"""Problems where waves of their own and 64 x 64 blocks are far apart, on operands that no cache holds: the default is
not behind the blocks, whichever it takes."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_block_choice_gpu import TORCH, _operand

pytestmark = pytest.mark.gpu

VT, AX, MO = cc.ValueType, cc.ComplexAxisLocation, cc.MemOrder
FOOTPRINT = 640 << 20   # what passes touch before the same buffers come round


@pytest.mark.parametrize("tin,tout,layout,B,M,N,K", [
    (VT.float8e4m3, VT.float32, "pairs", 22, 32, 476, 2160),   # a second wave on few of the units
    (VT.float16, VT.float16, "pairs", 33, 384, 32, 1488),
    (VT.float16, VT.float32, "pairs", 104, 28, 128, 1360),
    (VT.float16, VT.float32, "planar", 197, 24, 49, 2992),     # as much memory as products
    (VT.int1, VT.int32, "planar", 126, 87, 16, 1024),          # tiles in two rounds
    (VT.int1, VT.int32, "planar", 5, 1064, 128, 9600),         # ... in three
    (VT.int1, VT.int32, "planar", 18, 128, 256, 17280),
    (VT.float16, VT.float32, "planar", 1, 256, 256, 2048),     # (waves by a factor of two)
])
def test_default_is_not_behind_64x64_blocks(tin, tout, layout, B, M, N, K):
    """At most 12 % (best of five alternations), as test_block_choice_gpu.py for the block shapes."""
    bits = {VT.float16: 16, VT.float8e4m3: 8, VT.int1: 1}[tin]
    sizes = [(B * 2 * rows * K * bits // 8 + 511) // 512 * 512 for rows in (M, N)] + [B * 2 * M * N * 4]
    slots = max(1, FOOTPRINT // sum(sizes))
    a, b = (_operand(slots * size * 8 // bits, tin) for size in sizes[:2])
    c = torch.zeros(slots * sizes[2] // 4, device="cuda")
    where = [[x.data_ptr() + i * size for x, size in zip((a, b, c), sizes)] for i in range(slots)]
    runs = {}
    for tile in (0, 4):
        with cc.option(cc.Option.gemm_block_tile, tile), cc.option(cc.Option.pipeline_route, 1):
            if layout == "pairs":
                runs[tile] = cc.Pipeline(B, M, N, K, 0, stream(), AX.complex_interleaved, AX.complex_planar,
                                         MO.row_major, MO.col_major, MO.row_major, tin, tout, cc.Variant.opt)
                assert runs[tile].ReadsInPlace()
            else:
                runs[tile] = cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, tout), cc.Variant.basic)
    best, at = dict.fromkeys(runs, float("inf")), 0
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(5):
        for tile, run in runs.items():
            e0.record()
            for _ in range(40):
                at = (at + 1) % slots
                run.Run(*where[at])
            e1.record()
            e1.synchronize()
            best[tile] = min(best[tile], e0.elapsed_time(e1) / 40 * 1e3)
    print("us: default %.1f, 64x64 %.1f" % (best[0], best[4]), flush=True)
    assert best[0] <= 1.12 * best[4], best
