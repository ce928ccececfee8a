"""A C that the last-level cache holds is still there for the kernel that reads it next."""
import statistics

import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TORCH = {VT.bfloat16: torch.bfloat16, VT.float8e4m3: torch.float8_e4m3fn}


@pytest.mark.parametrize("tin,axis,B,M,N,K", [
    (VT.bfloat16, PLANAR, 24, 1024, 1024, 256),          # 192 MiB of C
    (VT.float8e4m3, INTERLEAVED, 16, 1024, 1024, 256),   # 128 MiB
])
def test_reading_c_after_the_product(tin, axis, B, M, N, K):
    """The reader behind the default's blocks against the reader behind 64 x 64 blocks, whose stores are ordinary
    ones whatever the size (at most 1.2 times; stored past the caches 1.4 times and more)."""
    a, b = (torch.randn(B * 2 * rows * K, device="cuda").to(TORCH[tin]) for rows in (M, N))
    c = torch.zeros(B * 2 * M * N, device="cuda")
    pipes = {}
    for tile in (0, 4):
        with cc.option(cc.Option.gemm_block_tile, tile):
            pipes[tile] = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, VT.float32,
                                      cc.Variant.opt)
    times = {tile: [] for tile in pipes}
    for _ in range(15):
        for tile, pipe in pipes.items():
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.amax(c)
            pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
            e0.record()
            torch.amax(c)
            e1.record()
            e1.synchronize()
            times[tile].append(e0.elapsed_time(e1))
    reader = {tile: statistics.median(v) for tile, v in times.items()}
    assert reader[0] <= 1.2 * reader[4], reader
