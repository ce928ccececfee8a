"""KernelName tells apart the kernels that a size alone chooses between."""
import pytest

import ccglib_amd as cc
from gpu_util import stream

pytestmark = pytest.mark.gpu

VT = cc.ValueType


def name(tin, tout, B, M, N, K, variant=cc.Variant.opt, block_tile=0):
    with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.basic_retile, 0):
        return cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, tout), variant).KernelName()


@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
def test_int1_waves_that_share_k(variant):
    assert "by four waves along K" in name(VT.int1, VT.int32, 1, 512, 512, 2048, variant)
    assert "by four waves along K" in name(VT.int1, VT.int32, 3, 256, 512, 2048, variant, 5)    # 384 tiles of 32 x 32
    for case in ((1, 512, 512, 512), (7, 256, 512, 2048)):   # one K tile; 896 tiles
        got = name(VT.int1, VT.int32, *case, variant, 5)
        assert "32x32 a wave" in got and "along K" not in got


@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
def test_waves_of_16_bit_blocks(variant):
    few, many = (256, 96, 96, 1024), (300, 96, 96, 1024)   # (a unit each; more blocks than units)
    assert "128x128 block of eight waves" in name(VT.float16, VT.float32, *few, variant, 2)
    assert "128x128 block, " in name(VT.float16, VT.float32, *many, variant, 2)
    assert "128x128 block, " in name(VT.float8e4m3, VT.float32, *few, variant, 2)
