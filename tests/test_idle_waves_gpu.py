"""16-bit blocks whose lower or right part lies beyond C: with waves that leave their products out (where most blocks
have some and K is long enough) and without."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TORCH = {VT.float16: torch.float16, VT.bfloat16: torch.bfloat16, VT.float32: torch.float32}


@pytest.mark.parametrize("tin,tout", [(VT.float16, VT.float32), (VT.float16, VT.float16), (VT.bfloat16, VT.bfloat16)])
@pytest.mark.parametrize("layout", ["tiled", "planar", "pairs"])
@pytest.mark.parametrize("c_axis", [PLANAR, INTERLEAVED])
@pytest.mark.parametrize("B,M,N,K,beta", [
    (2, 33, 300, 288, 0),            # a unit each, every block has idle waves (eight-wave 128 x 128 blocks: rows only)
    (1, 300, 40, 293, 0.5 - 1j),     # columns, ragged rows
    (1, 300, 300, 288, 0),           # ... only some of the blocks
    (140, 64, 300, 130, 0),          # more blocks than units, every one
    (100, 300, 129, 520, 0.25j),     # ... many of them, rows and columns
    (100, 300, 129, 128, 0),         # ... K too short
])
def test_same_bits_as_64x64_blocks(tin, tout, layout, c_axis, B, M, N, K, beta):
    gen = torch.Generator(device="cuda").manual_seed(4)
    a, b = (torch.randn(B * 2 * rows * K, device="cuda", generator=gen).to(TORCH[tin]) for rows in (M, N))
    start = torch.randn(B * 2 * M * N, device="cuda", generator=gen).to(TORCH[tout])
    results = []
    for block_tile in (4, 1, 2):
        with cc.option(cc.Option.gemm_block_tile, block_tile), \
                cc.option(cc.Option.pipeline_route, 2 if layout == "tiled" else 1):
            pipe = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED if layout == "pairs" else PLANAR, c_axis, ROW, COL,
                               ROW, tin, tout, cc.Variant.opt, 1.5j, beta)
        assert pipe.ReadsInPlace() == (layout != "tiled")
        c = start.clone()
        pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
        torch.cuda.synchronize()
        results.append(c)
    assert not torch.equal(results[0], start)
    assert torch.equal(results[0], results[1])
    assert torch.equal(results[0], results[2])
