"""C rows of any length at any element-aligned address: the kernels store (and, with beta,
read) whole pieces of a row wherever they start. The result is the oracle's, and nothing
outside C changes."""
import numpy as np
import pytest
import torch

import ccglib_amd as cc
import oracle as orc
from gpu_util import (ORC_TYPE, check_float, dequantize, quantize, stream, to_device, to_host,
                      transpose_operand)

pytestmark = pytest.mark.gpu

VT, AX, MO = cc.ValueType, cc.ComplexAxisLocation, cc.MemOrder
GUARD = 64      # elements on either side of C


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("nx", [1, 3, 66, 129, 255, 259])
@pytest.mark.parametrize("axis", [AX.complex_planar, AX.complex_interleaved])
@pytest.mark.parametrize("tin,tout", [(VT.float16, VT.float32), (VT.bfloat16, VT.bfloat16),
                                      (VT.float32, VT.float16), (VT.float8e4m3, VT.float32),
                                      (VT.int1, VT.int32)])
@pytest.mark.parametrize("block_tile", [0, 1, 2])
def test_c_rows_of_any_length_and_alignment(block_tile, tin, tout, axis, nx, offset):
    B, ny, K = 2, 70, 64
    beta = 0.5 - 0.25j if (nx + offset) % 2 and tout != VT.int32 else 0
    rng = np.random.default_rng(nx)
    if tin == VT.int1:
        qa = rng.integers(0, 2 ** 32, B * 2 * ny * K // 32, dtype=np.uint32)
        qb = rng.integers(0, 2 ** 32, B * 2 * nx * K // 32, dtype=np.uint32)
    else:
        qa = quantize(rng.uniform(-1, 1, (B, 2, ny, K)).astype(np.float32), tin).reshape(-1)
        qb = quantize(rng.uniform(-1, 1, (B, 2, nx, K)).astype(np.float32), tin).reshape(-1)
    n = B * 2 * ny * nx
    dtype = {VT.float32: np.float32, VT.int32: np.int32}.get(tout, np.uint16)
    store = (lambda x: x if dtype == np.float32 else quantize(x, tout))
    if dtype == np.int32:
        buffer = rng.integers(-9, 9, n + 2 * GUARD).astype(np.int32)
    else:
        buffer = store(rng.uniform(0, 1, n + 2 * GUARD).astype(np.float32)).reshape(-1)
    c_in = buffer[GUARD + offset:GUARD + offset + n].copy()
    d = to_device(buffer)
    d_a, d_b = transpose_operand(qa, B, ny, K, tin), transpose_operand(qb, B, nx, K, tin)
    with cc.option(cc.Option.gemm_block_tile, block_tile):
        gemm = cc.GEMM(B, ny, nx, K, 0, stream(), cc.Precision(tin, tout), cc.Variant.opt, axis,
                       MO.row_major, MO.row_major, MO.col_major, 1, beta)
    gemm.Run(d_a.data_ptr(), d_b.data_ptr(),
             d.data_ptr() + (GUARD + offset) * np.dtype(dtype).itemsize)
    torch.cuda.synchronize()
    after = to_host(d, dtype)
    assert np.array_equal(after[:GUARD + offset], buffer[:GUARD + offset])
    assert np.array_equal(after[GUARD + offset + n:], buffer[GUARD + offset + n:])
    got = after[GUARD + offset:GUARD + offset + n]
    planes = (lambda c: np.ascontiguousarray(c.reshape(B, ny, nx, 2).transpose(0, 3, 1, 2))
              if axis == AX.complex_interleaved else c.reshape(B, 2, ny, nx))
    got, c_in = planes(got), planes(c_in)
    want = orc.gemm(qa, qb, ny, nx, K, ORC_TYPE[tin], ORC_TYPE[tout], int(MO.row_major), 1, beta,
                    c_in.reshape(-1) if beta else None)
    if tin == VT.int1:
        assert np.array_equal(got, want.reshape(got.shape))
        return
    want64 = orc.gemm_float64(qa, qb, ny, nx, K, ORC_TYPE[tin], int(MO.row_major))
    if beta:
        c64 = dequantize(c_in, tout).astype(np.float64)
        w = want64[:, 0] + 1j * want64[:, 1] + beta * (c64[:, 0] + 1j * c64[:, 1])
        want64 = np.stack([w.real, w.imag], axis=1)
    check_float(dequantize(got, tout), dequantize(want, tout).reshape(got.shape), want64, tin, tout)


@pytest.mark.parametrize("block_tile", [1, 2, 4])
@pytest.mark.parametrize("rows", ["planar", "interleaved"])
@pytest.mark.parametrize("tin,tout", [(VT.float16, VT.float16), (VT.bfloat16, VT.bfloat16),
                                      (VT.float16, VT.float32), (VT.float8e4m3, VT.float32)])
def test_c_rows_behind_planar_and_interleaved_operands(block_tile, rows, tin, tout):
    """The same for operands read in place. Blocks that regroup a wave's 64 x 64 results through LDS
    (256 x 128 on interleaved rows, the two larger ones of 8-bit input) store 16 bytes wherever a row
    starts (every first wave here lies inside C), the others store from registers; with a complex
    alpha where C is offset."""
    B, ny, K = 2, 70, 64
    dtype = np.float32 if tout == VT.float32 else np.uint16
    for nx in (66, 129, 255):
        rng = np.random.default_rng(nx)
        qa = quantize(rng.uniform(-1, 1, (B, 2, ny, K)).astype(np.float32), tin)
        qb = quantize(rng.uniform(-1, 1, (B, 2, nx, K)).astype(np.float32), tin)
        want64 = orc.gemm_float64(qa.reshape(-1), qb.reshape(-1), ny, nx, K, ORC_TYPE[tin], int(MO.row_major))
        if rows == "interleaved":
            d_a, d_b = (to_device(np.ascontiguousarray(q.transpose(0, 2, 3, 1))) for q in (qa, qb))
        else:
            d_a, d_b = to_device(qa), to_device(qb)
        for offset in (0, 1):
            alpha = 0.5 - 1.5j if offset else 1
            n = B * 2 * ny * nx
            fill = rng.uniform(0, 1, n + 2 * GUARD).astype(np.float32)
            buffer = fill if tout == VT.float32 else quantize(fill, tout).reshape(-1)
            d = to_device(buffer)
            with cc.option(cc.Option.gemm_block_tile, block_tile), cc.option(cc.Option.pipeline_route, 1):
                if rows == "interleaved":
                    run = cc.Pipeline(B, ny, nx, K, 0, stream(), AX.complex_interleaved, AX.complex_planar,
                                      MO.row_major, MO.col_major, MO.row_major, tin, tout, cc.Variant.opt, alpha)
                    assert run.ReadsInPlace()
                else:
                    run = cc.GEMM(B, ny, nx, K, 0, stream(), cc.Precision(tin, tout), cc.Variant.basic,
                                  alpha=alpha)
            run.Run(d_a.data_ptr(), d_b.data_ptr(),
                    d.data_ptr() + (GUARD + offset) * np.dtype(dtype).itemsize)
            torch.cuda.synchronize()
            after = to_host(d, dtype)
            assert np.array_equal(after[:GUARD + offset], buffer[:GUARD + offset])
            assert np.array_equal(after[GUARD + offset + n:], buffer[GUARD + offset + n:])
            got = after[GUARD + offset:GUARD + offset + n].reshape(B, 2, ny, nx)
            want = orc.gemm(qa.reshape(-1), qb.reshape(-1), ny, nx, K, ORC_TYPE[tin], ORC_TYPE[tout],
                            int(MO.row_major), alpha, 0, None)
            w = (want64[:, 0] + 1j * want64[:, 1]) * alpha
            check_float(dequantize(got, tout), dequantize(want, tout).reshape(got.shape),
                        np.stack([w.real, w.imag], axis=1), tin, tout)
