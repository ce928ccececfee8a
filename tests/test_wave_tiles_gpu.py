"""Small problems run on waves that share nothing, each with a tile of 16 x 16, 32 x 16 or 32 x 32 elements
of C and a ring of its own of 8, 5 or 4 K tiles."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW, float_case, int1_case

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TORCH = {VT.float16: torch.float16, VT.bfloat16: torch.bfloat16, VT.float32: torch.float32,
         VT.float8e4m3: torch.float8_e4m3fn, VT.float8e5m2: torch.float8_e5m2}
PER_TILE = {VT.float16: 32, VT.bfloat16: 32, VT.float8e4m3: 64, VT.float8e5m2: 64}


@pytest.mark.parametrize("block_tile", [5, 6, 7])
@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("tin,tout", [(VT.float16, VT.float32), (VT.float16, VT.float16),
                                      (VT.bfloat16, VT.bfloat16), (VT.float8e4m3, VT.float32),
                                      (VT.float8e5m2, VT.float32)])
def test_against_the_oracle(block_tile, variant, tin, tout):
    with cc.option(cc.Option.gemm_block_tile, block_tile):
        gemm = cc.GEMM(1, 33, 17, 40, 0, stream(), cc.Precision(tin, tout), variant)
        assert "complex_gemm_mfma_wave" in gemm.KernelName()
        float_case(1, 33, 17, 40, tin, tout, variant, PLANAR, ROW, seed=1)
        float_case(3, 16, 129, 330, tin, tout, variant, PLANAR, COL, alpha=0.5 - 1.5j, beta=0.25 + 0.5j, seed=2)
        if variant == cc.Variant.opt:
            float_case(2, 65, 31, 700, tin, tout, variant, INTERLEAVED, ROW, alpha=1.5j, beta=0.5, seed=3)


@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 128), (2, 33, 65, 1152), (1, 70, 30, 2560), (3, 32, 64, 4224),
                                     (1, 40, 20, 16384), (5, 256, 250, 16256), (9, 250, 256, 2688)])
def test_int1(variant, B, M, N, K):
    """One K tile; three to nine and 32 of them, which four waves share out unevenly, the last one partial; more tiles of C
    (320, 576) than units, two or three of them one after the other."""
    with cc.option(cc.Option.gemm_block_tile, 5):
        int1_case(B, M, N, K, variant, seed=1)
        int1_case(B, M, N, K, variant, c_order=COL, alpha=2 - 1j, beta=1 + 3j, seed=2)


@pytest.mark.parametrize("axis", [PLANAR, INTERLEAVED])
@pytest.mark.parametrize("tin", list(PER_TILE))
@pytest.mark.parametrize("tiles", [1, 3, 4, 5, 6, 7, 8, 9, 10, 11, 17])
@pytest.mark.parametrize("over", [0, -1, -8, 9])
def test_same_bits_as_64x64_blocks(axis, tin, tiles, over):
    """Rows in place, K at, one and eight below and nine above a number of whole K tiles around the
    lengths of the rings; rows of A and B one short of a tile, one over, and buffers at an odd address."""
    K = tiles * PER_TILE[tin] + over
    B, M, N = 2, 47, 33
    gen = torch.Generator(device="cuda").manual_seed(tiles * 10 + over)
    a, b = (torch.randn(B * 2 * rows * K + 1, device="cuda", generator=gen).to(TORCH[tin])[1:] for rows in (M, N))
    results = {}
    for block_tile in (4, 5, 6, 7):
        with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, 1), \
                cc.option(cc.Option.basic_retile, 0):
            if axis == INTERLEAVED:
                run = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, VT.float32,
                                  cc.Variant.opt)
            else:
                run = cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, VT.float32), cc.Variant.basic)
        c = torch.full((B, 2, M, N), float("nan"), device="cuda")
        a2, b2 = (a, b) if K % 16 else (a.clone(), b.clone())   # (whole chunks are read in place at whole addresses)
        run.Run(a2.data_ptr(), b2.data_ptr(), c.data_ptr())
        torch.cuda.synchronize()
        results[block_tile] = c
    assert not torch.isnan(results[4]).any()
    for block_tile in (5, 6, 7):
        assert torch.equal(results[4], results[block_tile]), block_tile


def test_choice():
    """Few tiles go to waves, the fewer the smaller; many to blocks; 32-bit input and forced shapes never."""
    def name(B, M, N, K, tin=VT.float16):
        return cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, VT.float32), cc.Variant.opt).KernelName()

    assert "16x16 a wave" in name(1, 256, 256, 256)
    assert "32x32 a wave" in name(1, 256, 256, 256, VT.float8e4m3)
    assert "_wave" not in name(64, 512, 4096, 576)
    assert "_wave" not in name(1, 256, 256, 256, VT.float32)
    with cc.option(cc.Option.gemm_block_tile, 4):
        assert "64x64 block" in name(1, 256, 256, 256)
