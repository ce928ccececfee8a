"""GPU parity tests of GEMMs and pipelines that read rows of any length in place: rows that end
inside a 16-byte chunk, at every remainder, from any address, against the bits of the tiled
route (planar rows: same arithmetic) or the oracle ((re, im) rows)."""
import numpy as np
import pytest
import torch

import ccglib_amd as cc
import oracle as orc
from gpu_util import (ORC_TYPE, check_float, dequantize, quantize, stream, to_device, to_host,
                      transpose_operand)

pytestmark = pytest.mark.gpu
VT = cc.ValueType
PLANAR, INTERLEAVED = cc.ComplexAxisLocation.complex_planar, cc.ComplexAxisLocation.complex_interleaved
ROW, COL = cc.MemOrder.row_major, cc.MemOrder.col_major

# (type, K): the shortest rows, one K tile and one element less and more, several K tiles, all
# remainders of a chunk among them
PLANAR_K = [(VT.float16, k) for k in (9, 15, 31, 33, 61, 66, 100, 229)] + \
           [(VT.bfloat16, 301), (VT.float32, 5), (VT.float32, 47), (VT.float32, 114)] + \
           [(VT.float8e4m3, k) for k in (17, 31, 63, 65, 130, 135, 268)] + [(VT.float8e5m2, 201)]
PAIRS_K = [(VT.float16, k) for k in (5, 31, 33, 62, 67, 97, 230)] + [(VT.bfloat16, 225)] + \
          [(VT.float8e4m3, k) for k in (9, 63, 65, 130, 197)] + [(VT.float8e5m2, 332)]


def operands(rng, B, M, N, K, tin, scale=1.0):
    qa = quantize((scale * rng.uniform(-1, 1, B * 2 * M * K)).astype(np.float32), tin)
    qb = quantize((scale * rng.uniform(-1, 1, B * 2 * N * K)).astype(np.float32), tin)
    return qa, qb


def pairs(q, B, rows, K):
    return np.ascontiguousarray(q.reshape(B, 2, rows, K).transpose(0, 2, 3, 1)).reshape(-1)


def at_offset(q, skew):
    """A device buffer that ends with the data (whatever is read behind a row's end is not
    there), which starts `skew` elements behind a 16-byte boundary."""
    d = to_device(np.concatenate([np.zeros(skew, q.dtype), q]))
    return d, d.data_ptr() + skew * q.dtype.itemsize


@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("tin,K", PLANAR_K)
def test_planar_rows(block_tile, tin, K):
    B, M, N = 2, 150, 270
    skew = K % 3
    qa, qb = operands(np.random.default_rng(K), B, M, N, K, tin)
    (d_a, p_a), (d_b, p_b) = at_offset(qa, skew), at_offset(qb, skew)
    for order in (ROW, COL):
        d_c = to_device(np.full(B * 2 * M * N, np.nan, dtype=np.float32))
        with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.basic_retile, 0):
            g = cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, VT.float32), cc.Variant.basic,
                        PLANAR, order)
        g.Run(p_a, p_b, d_c.data_ptr())
        t_a, t_b = transpose_operand(qa, B, M, K, tin), transpose_operand(qb, B, N, K, tin)
        want = to_device(np.full(B * 2 * M * N, np.nan, dtype=np.float32))
        cc.GEMM(B, M, N, K, 0, stream(), cc.Precision(tin, VT.float32), cc.Variant.opt, PLANAR,
                order).Run(t_a.data_ptr(), t_b.data_ptr(), want.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(d_c, want)


@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("tin,K", PAIRS_K)
def test_pairs(block_tile, tin, K):
    B, M, N = 2, 150, 270
    qa, qb = operands(np.random.default_rng(K), B, M, N, K, tin)
    skew = 2 * (K % 3)
    (d_a, p_a), (d_b, p_b) = at_offset(pairs(qa, B, M, K), skew), at_offset(pairs(qb, B, N, K), skew)
    d_c = to_device(np.full(B * 2 * M * N, np.nan, dtype=np.float32))
    with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, 1):
        p = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED, INTERLEAVED, ROW, COL, ROW, tin, VT.float32,
                        cc.Variant.opt)
    assert p.ReadsInPlace()
    p.Run(p_a, p_b, d_c.data_ptr())
    torch.cuda.synchronize()
    got = to_host(d_c, np.float32).reshape(B, M, N, 2).transpose(0, 3, 1, 2)
    check_float(got, orc.gemm(qa, qb, M, N, K, ORC_TYPE[tin], orc.FLOAT32),
                orc.gemm_float64(qa, qb, M, N, K, ORC_TYPE[tin]), tin, VT.float32)


@pytest.mark.parametrize("block_tile,B,M,N", [(4, 70, 180, 190), (2, 256, 140, 130), (1, 300, 150, 200)])
@pytest.mark.parametrize("axis,tin,K", [(PLANAR, VT.float16, 13), (PLANAR, VT.float16, 77), (PLANAR, VT.bfloat16, 205),
                                        (PLANAR, VT.float32, 7), (PLANAR, VT.float32, 45),
                                        (PLANAR, VT.float8e4m3, 29), (PLANAR, VT.float8e5m2, 333),
                                        (INTERLEAVED, VT.float16, 9), (INTERLEAVED, VT.float16, 141),
                                        (INTERLEAVED, VT.float32, 3), (INTERLEAVED, VT.float32, 37),
                                        (INTERLEAVED, VT.float8e4m3, 61), (INTERLEAVED, VT.float8e4m3, 259)])
def test_more_tiles_than_blocks(block_tile, B, M, N, axis, tin, K):
    """Blocks that go on to further C tiles: K of one K tile and of several, the row ends of the one put
    right while the copies of the next are under way. Planar rows: the bits of the tiled route."""
    qa, qb = operands(np.random.default_rng(K), B, M, N, K, tin)
    if axis == INTERLEAVED:
        qa, qb = pairs(qa, B, M, K), pairs(qb, B, N, K)
    d_a, d_b = to_device(qa), to_device(qb)
    outs = []
    for route in (1, 2):
        with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, route):
            p = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, VT.float32, cc.Variant.opt)
        assert p.ReadsInPlace() == (route == 1)
        d_c = torch.full((B, 2, M, N), np.nan, device="cuda")
        p.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
        outs.append(d_c)
    torch.cuda.synchronize()
    if axis == PLANAR:
        assert torch.equal(outs[0], outs[1])
    else:
        # two orders of the same products. fp32 sums: 2 K roundings each, of partial sums that never exceed the
        # sum of the moduli, 2 K here; 8-bit ones: each within 6e-5 of the product in 64 bits
        # (test_64x64_blocks_on_interleaved_bytes)
        difference = (outs[0] - outs[1]).double()
        if tin == VT.float8e4m3:
            assert difference.norm() <= 2 * 6e-5 * outs[1].double().norm()
        else:
            assert difference.abs().max() <= 2 * 2.0 ** -24 * (2 * K) ** 2


@pytest.mark.parametrize("axis", [PLANAR, INTERLEAVED])
def test_infinities_at_the_end_of_a_row(axis):
    # The last elements of a row are fetched together with some before them, which must not
    # count twice: neither in a sum nor as 0 times an infinity.
    B, M, N, K, tin = 1, 70, 80, 45, VT.float16
    qa, qb = operands(np.random.default_rng(1), B, M, N, K, tin)
    a, b = qa.reshape(B, 2, M, K), qb.reshape(B, 2, N, K)
    inf = np.float16(np.inf).view(np.uint16)
    a[0, 0, 3, K - 7], a[0, 1, 66, K - 1], b[0, 0, 50, 37], b[0, 1, 79, 40] = inf, inf, inf, inf
    d_a = to_device(pairs(qa, B, M, K) if axis == INTERLEAVED else qa)
    d_b = to_device(pairs(qb, B, N, K) if axis == INTERLEAVED else qb)
    d_c = to_device(np.zeros(B * 2 * M * N, dtype=np.float32))
    with cc.option(cc.Option.pipeline_route, 1):
        p = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, VT.float32, cc.Variant.opt)
    p.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
    torch.cuda.synchronize()
    got = to_host(d_c, np.float32).reshape(2, M, N)
    x = dequantize(a, tin).astype(np.float64)[0]
    y = dequantize(b, tin).astype(np.float64)[0]
    with np.errstate(invalid="ignore"):
        want = np.stack([(x[0][:, None] * y[0] - x[1][:, None] * y[1]).sum(2),
                         (x[0][:, None] * y[1] + x[1][:, None] * y[0]).sum(2)])
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(got), kind(want))
    finite = np.isfinite(want)
    assert np.allclose(got[finite], want[finite], rtol=0, atol=1e-4)


@pytest.mark.parametrize("tin,tout", [(VT.float16, VT.float32), (VT.float16, VT.float16),
                                      (VT.float32, VT.float32), (VT.float8e4m3, VT.float32)])
@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("K", [64, 77])
def test_planar_rows_to_pairs(tin, tout, block_tile, K):
    # planar rows read in place with (re, im) pairs in C: the bits of the tiled route
    B, M, N = 2, 150, 270
    qa, qb = operands(np.random.default_rng(K), B, M, N, K, tin)
    d_a, d_b = to_device(qa), to_device(qb)
    outs = []
    for route in (1, 2):
        with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, route):
            p = cc.Pipeline(B, M, N, K, 0, stream(), PLANAR, INTERLEAVED, ROW, COL, ROW, tin, tout,
                            cc.Variant.opt, 0.5 + 2j, 0)
        assert p.ReadsInPlace() == (route == 1)
        d_c = torch.full((B * 2 * M * N,), -1, dtype=torch.float32 if tout == VT.float32 else torch.float16,
                         device="cuda")
        p.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
        outs.append(d_c)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("K", [2 ** 31 - 1, 2 ** 31 - 8])
def test_pairs_in_rows_of_4_gib(K):
    # Rows that end less than a K tile below 4 GiB, inside a chunk and behind one: the offset of the last
    # chunk's end has no 32 bits.
    M, tin = 2, VT.float8e4m3
    at = [0, 5, K - 9, K - 2, K - 1]
    a = np.array([[3 - 2j, 1j, 2, 5, 1 + 4j], [1, 2, 3 + 1j, 4j, -6]])
    b = np.array([2, 1 - 1j, 3 + 2j, 1j, 4 - 1j])
    d_a, d_b = (torch.zeros(rows * 2 * K, dtype=torch.uint8, device="cuda") for rows in (M, 1))
    for d, values in ((d_a, a), (d_b, b[None])):
        for row, v in enumerate(values):
            for k, z in zip(at, v):
                pair = torch.tensor([z.real, z.imag]).to(torch.float8_e4m3fn).view(torch.uint8)
                d[2 * (row * K + k):2 * (row * K + k) + 2] = pair.cuda()
    d_c = torch.full((2, M), np.nan, device="cuda")
    with cc.option(cc.Option.pipeline_route, 1):
        p = cc.Pipeline(1, M, 1, K, 0, stream(), INTERLEAVED, PLANAR, ROW, COL, ROW, tin, VT.float32, cc.Variant.opt)
    assert p.ReadsInPlace()
    p.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
    got = d_c.cpu().numpy()
    assert np.array_equal(got[0] + 1j * got[1], a @ b)
