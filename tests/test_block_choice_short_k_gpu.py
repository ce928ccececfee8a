"""The block shape of 16-bit problems with short K, and of pairs of C with beta, where a tile's stores count for more
than its products: the default is the fastest shape, or close to it."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_block_choice_gpu import TORCH, _operand, _time

pytestmark = pytest.mark.gpu

VT, AX = cc.ValueType, cc.ComplexAxisLocation


@pytest.mark.parametrize("tin,tout,layout,c_axis,beta,B,M,N,K", [
    (VT.bfloat16, VT.bfloat16, "pairs", AX.complex_interleaved, 0, 45, 320, 176, 112),
    (VT.float16, VT.float32, "pairs", AX.complex_interleaved, 0.5, 86, 192, 256, 80),
    (VT.bfloat16, VT.bfloat16, "pairs", AX.complex_interleaved, 0.5, 53, 673, 176, 208),
    (VT.float16, VT.float16, "pairs", AX.complex_interleaved, 0.5, 43, 144, 1024, 32),
    (VT.float16, VT.float32, "pairs", AX.complex_interleaved, 0.5, 225, 256, 165, 115),   # (ragged rows)
    (VT.bfloat16, VT.bfloat16, "pairs", AX.complex_planar, 0, 19, 192, 832, 80),
    (VT.float16, VT.float16, "planar", AX.complex_planar, 0.5, 60, 1536, 128, 80),
    (VT.float16, VT.float16, "planar", AX.complex_planar, 0, 4, 232, 2240, 32),
])
def test_default_block_shape_is_close_to_the_fastest(tin, tout, layout, c_axis, beta, B, M, N, K):
    """At most 12 % behind the fastest of the three shapes, as the problems of longer K (best of three alternations)."""
    a, b = (_operand(B * 2 * r * K, tin) for r in (M, N))
    c = torch.zeros(B * 2 * M * N, device="cuda", dtype=TORCH[tout])
    pipes = {}
    for tile in (0, 1, 2, 4):
        with cc.option(cc.Option.gemm_block_tile, tile), cc.option(cc.Option.pipeline_route, 1):
            pipes[tile] = cc.Pipeline(B, M, N, K, 0, stream(),
                                      AX.complex_interleaved if layout == "pairs" else AX.complex_planar, c_axis,
                                      cc.MemOrder.row_major, cc.MemOrder.col_major, cc.MemOrder.row_major, tin, tout,
                                      cc.Variant.opt, 1, beta)
            assert pipes[tile].ReadsInPlace()
    best = dict.fromkeys(pipes, float("inf"))
    for _ in range(3):
        for tile, pipe in pipes.items():
            best[tile] = min(best[tile], _time(pipe, a, b, c))
    print("us: " + ", ".join("%d %.1f" % v for v in best.items()), flush=True)
    assert best[0] <= 1.12 * min(best[1], best[2], best[4]), best
