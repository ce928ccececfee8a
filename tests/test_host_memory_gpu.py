"""Host-pointer Run on page-locked memory: one kernel fetches the operands and the GEMM stores C in
the caller's buffer, wherever that begins; the same bits as the device Run, and nothing around C changes."""
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW

pytestmark = pytest.mark.gpu

VT = cc.ValueType
TORCH = {VT.float16: torch.float16, VT.float32: torch.float32, VT.float8e4m3: torch.float8_e4m3fn}
GUARD = 64


@pytest.mark.parametrize("c_pinned", [True, False])
@pytest.mark.parametrize("offset_in,offset_out", [(0, 0), (3, 1), (16, 8)])   # (in and out in bytes of an element)
@pytest.mark.parametrize("beta", [0, 0.5 - 1j])
@pytest.mark.parametrize("tin,tout,axis,B,M,N,K", [
    (VT.float16, VT.float32, INTERLEAVED, 1, 1, 1, 8),          # less than one piece of the copy
    (VT.float16, VT.float16, PLANAR, 3, 33, 70, 61),
    (VT.float8e4m3, VT.float32, PLANAR, 2, 47, 19, 87),         # operands that end anywhere
    (VT.float8e4m3, VT.float32, INTERLEAVED, 1, 64, 64, 64),    # of 8 KiB: half a block of the copy
    (VT.float16, VT.float32, PLANAR, 1, 64, 128, 32),           # one block, two blocks exactly
    (VT.float32, VT.float32, INTERLEAVED, 1, 300, 257, 129),
    (VT.float16, VT.float32, INTERLEAVED, 1, 512, 1024, 576),   # 192 x 256 blocks, or what C's place allows
    (VT.float16, VT.float32, PLANAR, 1, 1024, 1100, 40),        # C of more than 8 MiB
])
def test_page_locked_memory(tin, tout, axis, B, M, N, K, beta, offset_in, offset_out, c_pinned):
    gen = torch.Generator().manual_seed(3)

    def place(x, offset, pinned=True):
        """x inside a larger buffer, `offset` elements behind GUARD ones."""
        buffer = torch.zeros(x.numel() + 2 * GUARD, dtype=x.dtype)
        buffer = buffer.pin_memory() if pinned else buffer
        view = buffer[GUARD + offset:GUARD + offset + x.numel()]
        view.copy_(x)
        return buffer, view

    a, b = (torch.randn(B * 2 * rows * K, generator=gen).to(TORCH[tin]) for rows in (M, N))
    c = torch.randn(B * 2 * M * N, generator=gen).to(TORCH[tout])
    pipe = cc.Pipeline(B, M, N, K, 0, stream(), axis, PLANAR, ROW, COL, ROW, tin, tout, cc.Variant.opt,
                       1, beta)
    d_a, d_b, d_c = a.cuda(), b.cuda(), c.cuda()
    pipe.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
    torch.cuda.synchronize()
    (_, h_a), (_, h_b), (c_buffer, h_c) = place(a, offset_in), place(b, offset_in), place(c, offset_out, c_pinned)
    for _ in range(2):
        h_c.copy_(c)
        pipe.RunHost(h_a.data_ptr(), h_b.data_ptr(), h_c.data_ptr())
        assert torch.equal(h_c, d_c.cpu())
    h_c.zero_()
    assert not c_buffer.any()
    assert torch.equal(h_a.view(torch.uint8), a.view(torch.uint8))
