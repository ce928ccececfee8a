"""Ragged rows of many K tiles that are read in place by default run on waves where 64 x 64 blocks are slower."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW
from test_pipeline_gpu import _time_runs

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TORCH = {VT.float16: torch.float16, VT.float8e4m3: torch.float8_e4m3fn}


@pytest.mark.parametrize("axis,tin,B,M,N,K", [
    (PLANAR, VT.float16, 55, 32, 16, 7026),
    (PLANAR, VT.float8e4m3, 100, 32, 16, 7027),
    (INTERLEAVED, VT.float16, 60, 16, 32, 3003),
])
def test_default_route(axis, tin, B, M, N, K):
    """In place, at least 1.5 times as fast as the blocks, the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(9)
    a, b = (torch.randn(B * 2 * rows * K, device="cuda", generator=gen).to(TORCH[tin]) for rows in (M, N))
    pipes, results, best = {}, {}, {}
    for tile in (0, 4):
        with cc.option(cc.Option.gemm_block_tile, tile):
            pipes[tile] = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, VT.float32,
                                      cc.Variant.opt)
        assert pipes[tile].ReadsInPlace()
        results[tile] = torch.full((B, 2, M, N), float("nan"), device="cuda")
        best[tile] = float("inf")
    for _ in range(3):
        for tile, pipe in pipes.items():
            best[tile] = min(best[tile], _time_runs(pipe, a, b, results[tile], budget_ms=10.0))
    print("ms: default %.4f, 64x64 %.4f" % (best[0], best[4]), flush=True)
    assert torch.equal(results[0], results[4])
    assert 1.5 * best[0] <= best[4], best


def test_basic_gemm():
    with cc.option(cc.Option.basic_retile, 0):
        gemm = cc.GEMM(1, 64, 320, 6598, 0, stream(), cc.Precision(VT.float16, VT.float32), cc.Variant.basic)
    assert "_wave" in gemm.KernelName()
