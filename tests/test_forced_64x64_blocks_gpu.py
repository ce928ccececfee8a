"""The 64 x 64 block kernel on problems that by default go to waves of their own: half an operand tile high, so blocks
start in the middle of one."""
import pytest

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW, float_case, int1_case
from test_small_blocks_gpu import TYPES

pytestmark = pytest.mark.gpu

VT = cc.ValueType


def kernel(B, M, N, K, tin, tout, variant):
    return cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, tout), variant).KernelName()


@pytest.mark.parametrize("tin,tout", TYPES)
@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("B,M,N,K", [
    (1, 1, 1, 16),         # one element, one K tile: the ring runs past the work
    (2, 64, 64, 64),       # one block exactly
    (2, 63, 65, 80),       # one short of a block, one more than one
    (1, 129, 190, 1040),   # blocks in both halves of an operand tile, the last one partial
    (3, 200, 320, 336),    # several blocks, more K tiles than ring slots
])
def test_float(B, M, N, K, tin, tout, variant):
    assert ("_wave" in kernel(B, M, N, K, tin, tout, variant)) == (tin != VT.float32)
    with cc.option(cc.Option.gemm_block_tile, 4):
        assert "64x64 block" in kernel(B, M, N, K, tin, tout, variant)
        float_case(B, M, N, K, tin, tout, variant, PLANAR, ROW, seed=1)
        float_case(B, M, N, K, tin, tout, variant, PLANAR, COL, alpha=0.5 - 1.5j, beta=0.25 + 0.5j, seed=2)
        if variant == cc.Variant.opt:
            float_case(B, M, N, K, tin, tout, variant, INTERLEAVED, ROW, alpha=1.5j, seed=3)
            float_case(B, M, N, K, tin, tout, variant, INTERLEAVED, COL, beta=0.5, seed=4)


@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 128), (2, 64, 64, 512), (2, 63, 65, 1152), (1, 129, 190, 4224)])
def test_int1(B, M, N, K, variant):
    assert "_wave" in kernel(B, M, N, K, VT.int1, VT.int32, variant)
    with cc.option(cc.Option.gemm_block_tile, 4):
        assert "64x64 block" in kernel(B, M, N, K, VT.int1, VT.int32, variant)
        int1_case(B, M, N, K, variant, seed=1)
        int1_case(B, M, N, K, variant, c_order=COL, alpha=2 - 1j, beta=1 + 3j, seed=2)
        if variant == cc.Variant.opt:
            int1_case(B, M, N, K, variant, c_axis=INTERLEAVED, seed=3)
