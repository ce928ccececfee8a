"""GPU tests of 32-bit input, whose values the kernels split into three bf16: accuracy of fp32
products over the whole range of the type, and infinities, NaN and sums beyond what the split
sums hold, on every block shape and operand layout."""
import numpy as np
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream, to_device, to_host, transpose_operand

pytestmark = pytest.mark.gpu
VT = cc.ValueType
PLANAR, INTERLEAVED = cc.ComplexAxisLocation.complex_planar, cc.ComplexAxisLocation.complex_interleaved
ROW, COL = cc.MemOrder.row_major, cc.MemOrder.col_major
LAYOUTS = ["tiled", "planar", "pairs"]


def product(layout, block_tile, a, b, beta=0, c=None):
    """C of planar a [B][2][M][K] and b [B][2][N][K]."""
    B, _, M, K = a.shape
    N = b.shape[2]
    d_c = to_device(np.full((B, 2, M, N), np.nan, np.float32) if c is None else c)
    with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, 1), \
            cc.option(cc.Option.basic_retile, 0):
        if layout == "pairs":
            obj = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED, PLANAR, ROW, COL, ROW, VT.float32, VT.float32,
                              cc.Variant.opt, 1, beta)
            assert obj.ReadsInPlace()
            d_a, d_b = (to_device(np.ascontiguousarray(x.transpose(0, 2, 3, 1))) for x in (a, b))
        else:
            variant = cc.Variant.opt if layout == "tiled" else cc.Variant.basic
            obj = cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(VT.float32, VT.float32), variant, beta=beta)
            d_a, d_b = ((transpose_operand(x.reshape(-1), B, x.shape[2], K, VT.float32)
                         if layout == "tiled" else to_device(x)) for x in (a, b))
    obj.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
    torch.cuda.synchronize()
    return to_host(d_c, np.float32).reshape(B, 2, M, N)


def exact(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64).transpose(0, 1, 3, 2)
    return np.stack([a[:, 0] @ b[:, 0] - a[:, 1] @ b[:, 1], a[:, 0] @ b[:, 1] + a[:, 1] @ b[:, 0]], 1)


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("K", [4, 5, 16, 17, 32, 47, 96, 333])
def test_accuracy(layout, block_tile, K):
    B, M, N = 2, 150, 290
    rng = np.random.default_rng(K)
    a = rng.standard_normal((B, 2, M, K)).astype(np.float32)
    b = rng.standard_normal((B, 2, N, K)).astype(np.float32)
    got, want = product(layout, block_tile, a, b), exact(a, b)
    # (wide enough for 12 roundings of the whole sum per 16 values of K, by up to 2^-24 of a partial
    # sum, which never exceeds the sum of the moduli; the next two tests are closer)
    scale = np.abs(a).astype(np.float64), np.abs(b).astype(np.float64).transpose(0, 1, 3, 2)
    moduli = np.stack([scale[0][:, 0] @ scale[1][:, 0] + scale[0][:, 1] @ scale[1][:, 1],
                       scale[0][:, 0] @ scale[1][:, 1] + scale[0][:, 1] @ scale[1][:, 0]], 1)
    assert np.all(np.abs(got - want) <= moduli * (2.0 ** -23 + 2.0 ** -24 * (12 * (K // 16 + 1) + 1)))
    # rounding errors of random sign: what fp32 products added up in fp32 show
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * (2 + 1.5 * np.sqrt(2 * K)) * np.linalg.norm(want)


def fp32_sum_error(n):
    """Relative error of n complex products added up in fp32: 2 n roundings of 0.42 * 2^-24 of the
    partial sum each in the mean, and with random signs the squares of the partial sums grow evenly,
    so together 0.42 * 2^-24 * sqrt((2 n + 1) / 2); a tenth more for the sample."""
    return 2.0 ** -24 * 0.33 * np.sqrt(2 * n + 1)


@pytest.mark.parametrize("block_tile", [2, 4])
@pytest.mark.parametrize("layout,K", [(layout, K) for layout in LAYOUTS for K in (1, 2, 3, 4, 5, 16, 17, 333)
                                      if (layout, K) != ("pairs", 1)])   # (rows of at least 16 bytes)
def test_no_less_accurate_than_fp32_sums(layout, block_tile, K):
    rng = np.random.default_rng(K)
    a = rng.standard_normal((2, 2, 150, K)).astype(np.float32)
    b = rng.standard_normal((2, 2, 290, K)).astype(np.float32)
    got, want = product(layout, block_tile, a, b), exact(a, b)
    assert np.linalg.norm(got - want) <= fp32_sum_error(K) * np.linalg.norm(want)


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [2, 4])
def test_two_products_a_row(layout, block_tile):
    M, N = 150, 290
    rng = np.random.default_rng(5)
    a = np.zeros((1, 2, M, 2 * M), np.float32)
    for first in (0, M):
        a[0, :, np.arange(M), first + rng.permutation(M)] = rng.standard_normal((M, 2))
    b = rng.standard_normal((1, 2, N, 2 * M)).astype(np.float32)
    got, want = product(layout, block_tile, a, b), exact(a, b)
    assert np.linalg.norm(got - want) <= fp32_sum_error(2) * np.linalg.norm(want)


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [2, 4])
def test_single_products_are_rounded_once(layout, block_tile):
    # a gain for every row: half a unit in the last place, and the seven small products' roundings,
    # 2^-24 of a sum below 2^-7 of the product each
    M, N = 150, 290
    rng = np.random.default_rng(5)
    a = np.zeros((1, 2, M, M), np.float32)
    a[0, 0, np.arange(M), rng.permutation(M)] = rng.standard_normal(M)
    b = rng.standard_normal((1, 2, N, M)).astype(np.float32)
    got, want = product(layout, block_tile, a, b), exact(a, b)
    assert np.all(np.abs(got - want) <= (0.5 + 7 * 2.0 ** -8) * np.spacing(np.abs(want).astype(np.float32)))


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("exponents", [(-126, 100), (100, -126), (-140, 120), (-60, -60), (39, 39)])
def test_every_magnitude_is_split_exactly(layout, block_tile, exponents):
    B, M, N, K = 1, 70, 90, 40
    rng = np.random.default_rng(7)
    a = np.ldexp(rng.standard_normal((B, 2, M, K)), exponents[0]).astype(np.float32)
    b = np.ldexp(rng.standard_normal((B, 2, N, K)), exponents[1]).astype(np.float32)
    got, want = product(layout, block_tile, a, b), exact(a, b)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("beta", [0, 0.5 - 0.25j])
def test_infinities_nan_and_large_sums(layout, block_tile, beta):
    B, M, N, K = 2, 140, 270, 50
    rng = np.random.default_rng(3)
    a = rng.standard_normal((B, 2, M, K)).astype(np.float32)
    b = rng.standard_normal((B, 2, N, K)).astype(np.float32)
    c = rng.standard_normal((B, 2, M, N)).astype(np.float32)
    a[0, 0, 3, 49], a[0, 1, 130, 0], b[0, 1, 200, 17] = np.inf, -np.inf, np.inf
    a[1, 0, 70, 5] = np.nan
    a[1, :, 20] *= np.float32(1e20)      # sums of 1e32, beyond those that the split sums hold
    b[1, :, 7] *= np.float32(1e12)
    a[0, 0, 64, 1], b[0, 0, 3, 1] = 3.3e38, 1.5      # overflows to infinity; rounds to infinity as bf16
    got = product(layout, block_tile, a, b, beta=beta, c=c)
    with np.errstate(invalid="ignore", over="ignore"):
        want = exact(a, b)
        if beta:
            z = beta * (c[:, 0].astype(np.complex128) + 1j * c[:, 1])
            want += np.stack([z.real, z.imag], 1)
        want = want.astype(np.float32)
    # (element a[0, 0, 64, 1] overflows where its product does: nothing but the sign is compared there)
    for kind in (np.isnan, np.isposinf, np.isneginf):
        same = kind(got) == kind(want)
        same[0, :, 64] = True
        assert np.all(same)
    assert np.isposinf(got[0, 0, 64, 3])
    finite = np.isfinite(want) & np.isfinite(got)
    x, y = (np.abs(np.nan_to_num(v, posinf=0, neginf=0)).astype(np.float64) for v in (a, b))
    bound = np.stack([x.sum(1) @ y.sum(1).transpose(0, 2, 1)] * 2, 1) + 2
    assert np.all(np.abs(got[finite].astype(np.float64) - want[finite]) <= 2.0 ** -18 * bound[finite])


def pipeline_product(layout, block_tile, a, b, c_axis=PLANAR, order=ROW, alpha=1, beta=0, tout=VT.float32, c=None):
    """C as [B][2][M][N] of planar a [B][2][M][K] and b [B][2][N][K], by a pipeline that reads planar
    rows or pairs in place or transposes them into tiles."""
    B, _, M, K = a.shape
    N = b.shape[2]
    dtype = {VT.float32: torch.float32, VT.float16: torch.float16, VT.bfloat16: torch.bfloat16}[tout]
    il = c_axis == INTERLEAVED
    if c is None:
        c = np.full((B, 2, M, N), np.nan, np.float32)
    d_c = torch.from_numpy(c).cuda().to(dtype)
    d_c = d_c.permute(0, 2, 3, 1) if il else d_c
    if order == COL:
        d_c = d_c.permute(0, 2, 1, 3) if il else d_c.permute(0, 1, 3, 2)
    d_c = d_c.contiguous()
    axis = INTERLEAVED if layout == "pairs" else PLANAR
    d_a, d_b = (to_device(np.ascontiguousarray(x.transpose(0, 2, 3, 1)) if layout == "pairs" else x) for x in (a, b))
    with cc.option(cc.Option.gemm_block_tile, block_tile), \
            cc.option(cc.Option.pipeline_route, 2 if layout == "tiled" else 1):
        p = cc.Pipeline(B, M, N, K, 0, stream(), axis, c_axis, ROW, COL, order, VT.float32, tout, cc.Variant.opt,
                        alpha, beta)
    assert p.ReadsInPlace() == (layout != "tiled")
    p.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
    torch.cuda.synchronize()
    if order == COL:
        d_c = d_c.permute(0, 2, 1, 3) if il else d_c.permute(0, 1, 3, 2)
    return (d_c.permute(0, 3, 1, 2) if il else d_c).float().cpu().numpy()


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [2, 4])
@pytest.mark.parametrize("B,M,N,K", [(2, 150, 270, 16), (2, 150, 270, 333), (200, 150, 140, 45), (300, 33, 260, 7)])
def test_nan_in_rows(layout, block_tile, B, M, N, K):
    """NaN among the samples (no infinities): every sum of such a row is NaN, and all others have the bits
    that they have without - also those that the same blocks compute next (the larger batches)."""
    rng = np.random.default_rng(B + K)
    a = rng.standard_normal((B, 2, M, K)).astype(np.float32)
    b = rng.standard_normal((B, 2, N, K)).astype(np.float32)
    clean = pipeline_product(layout, block_tile, a, b)
    for x in (a, b):   # a few rows of most matrices, and every row of one
        for i in range(0, B, 3 if x is a else 4):
            for r in rng.integers(0, x.shape[2], 2):
                x[i, rng.integers(2), r, rng.integers(K)] = np.nan
    a[1, rng.integers(0, 2, M), np.arange(M), rng.integers(0, K, M)] = np.nan
    a[0, 0, M - 1, K - 1] = b[0, 1, N - 1, K - 1] = np.nan
    got = pipeline_product(layout, block_tile, a, b)
    rows, cols = np.isnan(a).any(axis=(1, 3)), np.isnan(b).any(axis=(1, 3))
    nan = (rows[:, :, None] | cols[:, None, :])[:, None] & np.ones((1, 2, 1, 1), bool)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan], clean[~nan])


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("block_tile", [2, 4])
@pytest.mark.parametrize("c_axis,order,alpha,beta,tout", [(PLANAR, COL, 1, 0, VT.float32),
                                                          (INTERLEAVED, ROW, 0.5 - 2j, 0, VT.float32),
                                                          (INTERLEAVED, COL, 1, 0.5 + 1j, VT.float32),
                                                          (PLANAR, ROW, 2, 0, VT.bfloat16),
                                                          (INTERLEAVED, ROW, 1, 0.25, VT.float16)])
def test_infinities_and_nan_before_further_tiles(layout, block_tile, c_axis, order, alpha, beta, tout):
    """More tiles than blocks, with infinities and NaN in the same wave's rows, in all forms of C."""
    B, M, N, K = 200, 150, 140, 37
    rng = np.random.default_rng(4)
    a = rng.standard_normal((B, 2, M, K)).astype(np.float32)
    b = rng.standard_normal((B, 2, N, K)).astype(np.float32)
    c = rng.integers(-8, 8, (B, 2, M, N)).astype(np.float32)
    for i in range(0, B, 5):
        a[i, 0, rng.integers(M), rng.integers(K)] = np.inf
        b[i, 1, rng.integers(N), rng.integers(K)] = -np.inf
        a[i, 1, rng.integers(M), rng.integers(K)] = np.nan
    got = pipeline_product(layout, block_tile, a, b, c_axis, order, alpha, beta, tout, c)
    # (no square of a sum overflows: where both parts are finite so is the result)
    with np.errstate(invalid="ignore"):
        re, im = exact(a, b).transpose(1, 0, 2, 3)
        # (alpha and beta part by part: in numpy's complex product an infinite part spoils the other)
        z, w = complex(alpha), complex(beta)
        want = np.stack([z.real * re - z.imag * im + w.real * c[:, 0] - w.imag * c[:, 1] if z.imag else
                         z.real * re + w.real * c[:, 0] - w.imag * c[:, 1],
                         z.imag * re + z.real * im + w.imag * c[:, 0] + w.real * c[:, 1] if z.imag else
                         z.real * im + w.imag * c[:, 0] + w.real * c[:, 1]], 1)
    finite = np.isfinite(want).all(axis=1, keepdims=True) & np.ones((1, 2, 1, 1), bool)
    assert not np.isfinite(got[~finite]).all(axis=None) and np.isfinite(got[finite]).all()
    if alpha == 1:   # (otherwise 0 times an infinity comes in)
        for kind in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(kind(got), kind(want))
    # 2 K roundings by half a unit of partial sums below 40 (five standard deviations), times alpha, and one to
    # the type of C
    unit = {VT.float32: 0.0, VT.float16: 2.0 ** -11, VT.bfloat16: 2.0 ** -8}[tout]
    difference = np.abs(got[finite] - want[finite])
    assert np.all(difference <= 2 * K * 2.0 ** -23 * 40 + 2 * unit * np.abs(want[finite]) + 1e-6)
