"""Problems that leave compute units without work at the larger block shapes run on 64 x 64
blocks: half an operand tile high, so blocks start in the middle of one."""
import numpy as np
import pytest

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW, float_case, int1_case, quantize, run_gemm

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TYPES = [(VT.float16, VT.float32), (VT.float16, VT.float16), (VT.bfloat16, VT.bfloat16),
         (VT.float32, VT.float32), (VT.float8e4m3, VT.float32), (VT.float8e5m2, VT.float32)]


def takes_64(B, M, N, K, tin, tout, variant):
    gemm = cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, tout), variant)
    return "64x64" in gemm.KernelName()


@pytest.mark.parametrize("tin,tout", TYPES)
@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("B,M,N,K", [
    (1, 1, 1, 16),         # one element, one K tile: the ring runs past the work
    (2, 64, 64, 64),       # one block exactly
    (2, 63, 65, 80),       # one short of a block, one more than one
    (1, 129, 190, 1040),   # blocks in both halves of an operand tile, the last one partial
    (3, 200, 320, 336),    # several blocks, more K tiles than ring slots
])
def test_64x64_blocks(B, M, N, K, tin, tout, variant):
    assert takes_64(B, M, N, K, tin, tout, variant)
    float_case(B, M, N, K, tin, tout, variant, PLANAR, ROW, seed=1)
    float_case(B, M, N, K, tin, tout, variant, PLANAR, COL, alpha=0.5 - 1.5j, beta=0.25 + 0.5j, seed=2)
    if variant == cc.Variant.opt:
        float_case(B, M, N, K, tin, tout, variant, INTERLEAVED, ROW, alpha=1.5j, seed=3)
        float_case(B, M, N, K, tin, tout, variant, INTERLEAVED, COL, beta=0.5, seed=4)


@pytest.mark.parametrize("tin,B,M,N,K", [(VT.float32, 70, 180, 190, 48), (VT.float16, 256, 33, 130, 64),
                                         (VT.float16, 256, 33, 130, 200), (VT.float8e4m3, 512, 60, 40, 64)])
def test_64x64_blocks_several_tiles_each(tin, B, M, N, K):
    """More tiles than resident blocks, among them K of one tile: the same bits as the
    128 x 128 block, which adds up in the same order."""
    rng = np.random.default_rng(5)
    qa = quantize(rng.uniform(-1, 1, (B, 2, M, K)).astype(np.float32), tin).reshape(-1)
    qb = quantize(rng.uniform(-1, 1, (B, 2, N, K)).astype(np.float32), tin).reshape(-1)
    for variant in (cc.Variant.basic, cc.Variant.opt):
        assert takes_64(B, M, N, K, tin, VT.float32, variant)
        got = run_gemm(qa, qb, B, M, N, K, tin, VT.float32, variant, alpha=0.5 - 2j)
        with cc.option(cc.Option.gemm_block_tile, 2):
            want = run_gemm(qa, qb, B, M, N, K, tin, VT.float32, variant, alpha=0.5 - 2j)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("tin,tout", TYPES[:3])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 3, 8), (2, 63, 65, 72), (200, 100, 40, 200), (256, 64, 130, 40)])
def test_64x64_blocks_on_interleaved_rows(B, M, N, K, tin, tout):
    """The pipeline's (re, im) rows of 16-bit samples, read in place."""
    import torch
    rng = np.random.default_rng(6)
    a = rng.uniform(-1, 1, (B, M, K, 2)).astype(np.float32)
    b = rng.uniform(-1, 1, (B, N, K, 2)).astype(np.float32)
    tdt = torch.float16 if tin == VT.float16 else torch.bfloat16
    d_a, d_b = torch.from_numpy(a).cuda().to(tdt), torch.from_numpy(b).cuda().to(tdt)
    results = []
    for block_tile in (4, 2):
        c = torch.full((B, 2, M, N), float("nan"), device="cuda",
                       dtype={VT.float32: torch.float32, VT.float16: torch.float16,
                              VT.bfloat16: torch.bfloat16}[tout])
        with cc.option(cc.Option.gemm_block_tile, block_tile):
            pipe = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED, PLANAR, ROW, COL, ROW, tin, tout,
                               cc.Variant.opt)
        assert pipe.ReadsInPlace()
        pipe.Run(d_a.data_ptr(), d_b.data_ptr(), c.data_ptr())
        torch.cuda.synchronize()
        results.append(c)
    assert torch.equal(results[0], results[1])
    ca = torch.view_as_complex(d_a.cpu().double()).numpy()
    cb = torch.view_as_complex(d_b.cpu().double()).numpy()
    want = np.einsum("bmk,bnk->bmn", ca, cb)
    got = results[0].cpu().double().numpy()
    got = got[:, 0] + 1j * got[:, 1]
    # fp32 sums of 2 K products, then one rounding to the type of C
    eps = {VT.float32: 0.0, VT.float16: 2.0 ** -11, VT.bfloat16: 2.0 ** -8}[tout]
    sums = np.einsum("bmk,bnk->bmn", np.abs(ca), np.abs(cb))
    assert (np.abs(got - want) <= 2 * K * 2.0 ** -23 * sums + 2 * eps * np.abs(want) + 1e-7).all()


@pytest.mark.parametrize("variant", [cc.Variant.basic, cc.Variant.opt])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 128), (2, 64, 64, 512), (2, 63, 65, 1152), (1, 129, 190, 4224),
                                     (70, 180, 190, 640)])   # (the last: several tiles a block)
def test_64x64_blocks_int1(B, M, N, K, variant):
    assert takes_64(B, M, N, K, VT.int1, VT.int32, variant)
    int1_case(B, M, N, K, variant, seed=1)
    int1_case(B, M, N, K, variant, c_order=COL, alpha=2 - 1j, beta=1 + 3j, seed=2)
    if variant == cc.Variant.opt:
        int1_case(B, M, N, K, variant, c_axis=INTERLEAVED, seed=3)


@pytest.mark.parametrize("axis", [PLANAR, INTERLEAVED])
@pytest.mark.parametrize("offsets", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 7, 32), (3, 129, 40, 544), (2, 8, 300, 1024)])
def test_packing_of_both_operands(B, M, N, K, offsets, axis):
    """Raw samples at any address: both operands in one launch, or one each where only one of them
    is aligned; row counts below, at and above a block of rows and a row tile."""
    import torch
    rng = np.random.default_rng(7)
    planes, device = [], []
    for rows, offset in ((M, offsets[0]), (N, offsets[1])):
        x = rng.integers(0, 2, (B, 2, rows, K), dtype=np.uint8)
        planes.append(2 * x.astype(np.int64) - 1)
        raw = np.ascontiguousarray(x if axis == PLANAR else x.transpose(0, 2, 3, 1)).reshape(-1)
        buffer = torch.zeros(raw.size + 16, dtype=torch.uint8, device="cuda")
        buffer[offset:offset + raw.size] = torch.from_numpy(raw).cuda()
        device.append(buffer)
    c = torch.zeros((B, 2, M, N), dtype=torch.int32, device="cuda")
    pipe = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, VT.int1, VT.int32,
                       cc.Variant.opt)
    pipe.Run(device[0].data_ptr() + offsets[0], device[1].data_ptr() + offsets[1], c.data_ptr())
    torch.cuda.synchronize()
    (ar, ai), (br, bi) = [(p[:, 0], p[:, 1]) for p in planes]
    brt, bit = br.transpose(0, 2, 1), bi.transpose(0, 2, 1)
    want = np.stack([ar @ brt - ai @ bit, ar @ bit + ai @ brt], axis=1)
    assert np.array_equal(c.cpu().numpy(), want)


@pytest.mark.parametrize("tin", [VT.float8e4m3, VT.float8e5m2])
@pytest.mark.parametrize("B,M,N,K", [(1, 1, 3, 8), (2, 63, 65, 200), (200, 100, 40, 136), (256, 64, 64, 512)])
def test_64x64_blocks_on_interleaved_bytes(B, M, N, K, tin):
    """The pipeline's (re, im) rows of 8-bit samples: the same bits as the 128 x 128 block, and the
    product in 64 bits within what the matrix instruction's sums of 64 lose (four times the largest
    relative error, 1.5e-5, and the largest difference, 8.4e-5 of the root mean square, measured on
    8-bit products of K up to 8192)."""
    import torch
    tdt = torch.float8_e4m3fn if tin == VT.float8e4m3 else torch.float8_e5m2
    gen = torch.Generator().manual_seed(8)
    a = torch.randn((B, M, K, 2), generator=gen).to(tdt).cuda()
    b = torch.randn((B, N, K, 2), generator=gen).to(tdt).cuda()
    results = []
    for block_tile in (4, 2):
        c = torch.full((B, 2, M, N), float("nan"), device="cuda")
        with cc.option(cc.Option.gemm_block_tile, block_tile):
            pipe = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED, PLANAR, ROW, COL, ROW, tin, VT.float32,
                               cc.Variant.opt)
        assert pipe.ReadsInPlace()
        pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
        torch.cuda.synchronize()
        results.append(c)
    assert torch.equal(results[0], results[1])
    ca = torch.view_as_complex(a.cpu().double()).numpy()
    cb = torch.view_as_complex(b.cpu().double()).numpy()
    got = results[0].cpu().double().numpy()
    got = got[:, 0] + 1j * got[:, 1]
    want = np.einsum("bmk,bnk->bmn", ca, cb)
    rms = np.sqrt(np.mean(np.abs(want) ** 2))
    assert np.linalg.norm(got - want) <= 6e-5 * np.linalg.norm(want)
    assert (np.abs(got - want) <= 3.5e-4 * np.maximum(rms, np.abs(want))).all()


@pytest.mark.parametrize("tin,tout", TYPES[:3])
@pytest.mark.parametrize("c_axis", [PLANAR, INTERLEAVED])
@pytest.mark.parametrize("layout", ["tiled", "planar", "pairs"])
@pytest.mark.parametrize("M,N,K,beta", [(128, 128, 64, 0), (70, 200, 40, 0), (129, 65, 96, 0.5 - 1j)])
def test_128x128_blocks_of_four_waves(tin, tout, c_axis, layout, M, N, K, beta):
    """More 128 x 128 tiles than units, with waves that lie beyond C: the same bits as 64 x 64 blocks."""
    import torch
    B = 300
    if layout == "planar" and c_axis == INTERLEAVED:
        return   # (the basic variant has planar C only)
    types = {VT.float16: torch.float16, VT.bfloat16: torch.bfloat16, VT.float32: torch.float32}
    gen = torch.Generator(device="cuda").manual_seed(4)
    a, b = (torch.randn(B * 2 * rows * K, device="cuda", generator=gen).to(types[tin]) for rows in (M, N))
    start = torch.randn(B * 2 * M * N, device="cuda", generator=gen).to(types[tout])
    axis = INTERLEAVED if layout == "pairs" else PLANAR
    results = []
    for block_tile in (2, 4):
        with cc.option(cc.Option.gemm_block_tile, block_tile), \
                cc.option(cc.Option.pipeline_route, 2 if layout == "tiled" else 1):
            pipe = cc.Pipeline(B, M, N, K, 0, stream(), axis, c_axis, ROW, COL, ROW, tin, tout, cc.Variant.opt, 1.5j, beta)
        c = start.clone()
        pipe.Run(a.data_ptr(), b.data_ptr(), c.data_ptr())
        torch.cuda.synchronize()
        results.append(c)
    assert not torch.equal(results[0], start)
    assert torch.equal(results[0], results[1])
