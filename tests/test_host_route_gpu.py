"""Host-pointer Run: operands that change in place between two calls, in every kind of page-locked memory, and which way
the data goes."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import ccglib_amd as cc
from gpu_util import stream
from test_gemm_gpu import COL, INTERLEAVED, PLANAR, ROW

pytestmark = pytest.mark.gpu

VT = cc.ValueType
# hipHostMallocDefault, WriteCombined, Coherent, NonCoherent
FLAGS = [0x0, 0x4, 0x40000000, 0x80000000]


class HostMemory:
    """hipHostMalloc with flags, as a numpy array."""

    def __init__(self, hip, dtype, n, flags):
        self.hip, self.p = hip, ctypes.c_void_p()
        nbytes = n * np.dtype(dtype).itemsize
        assert hip.hipHostMalloc(ctypes.byref(self.p), ctypes.c_size_t(nbytes), ctypes.c_uint(flags)) == 0
        self.array = np.frombuffer((ctypes.c_char * nbytes).from_address(self.p.value), dtype=dtype)

    def free(self):
        self.array = None
        assert self.hip.hipHostFree(self.p) == 0


@pytest.mark.parametrize("flags", FLAGS)
@pytest.mark.parametrize("B,M,N,K,beta", [(1, 64, 64, 64, 0), (2, 130, 70, 333, 0), (1, 512, 1024, 576, 0),
                                          (2, 130, 70, 333, 0.5 - 1j)])
def test_operands_change_between_runs(flags, B, M, N, K, beta):
    """Every call sees what the buffers hold then: the bits of the device Run on the same values."""
    hip = ctypes.CDLL("libamdhip64.so")
    memory = [HostMemory(hip, np.float16, B * 2 * rows * K, flags) for rows in (M, N)]
    memory.append(HostMemory(hip, np.float32, B * 2 * M * N, flags))
    a, b, c = (m.array for m in memory)
    pipe = cc.Pipeline(B, M, N, K, 0, stream(), INTERLEAVED, PLANAR, ROW, COL, ROW, VT.float16, VT.float32,
                       cc.Variant.opt, 1, beta)
    rng = np.random.default_rng(5)
    for _ in range(4):
        a[:] = rng.standard_normal(a.size).astype(np.float16)
        b[:] = rng.standard_normal(b.size).astype(np.float16)
        c[:] = rng.standard_normal(c.size).astype(np.float32)
        d_a, d_b, d_c = (torch.from_numpy(x.copy()).cuda() for x in (a, b, c))
        pipe.Run(d_a.data_ptr(), d_b.data_ptr(), d_c.data_ptr())
        torch.cuda.synchronize()
        pipe.RunHost(memory[0].p.value, memory[1].p.value, memory[2].p.value)
        assert np.array_equal(c, d_c.cpu().numpy())
    del a, b, c
    for m in memory:
        m.free()


PROGRAM = """
import torch
from torch.profiler import profile, ProfilerActivity
import ccglib_amd as cc
AX, MO, VT = cc.ComplexAxisLocation, cc.MemOrder, cc.ValueType

def host_run(pinned_in, pinned_c, M, N, K, beta=0):
    pipe = cc.Pipeline(1, M, N, K, 0, torch.cuda.current_stream().cuda_stream, AX.complex_interleaved,
                       AX.complex_planar, MO.row_major, MO.col_major, MO.row_major, VT.float16, VT.float32,
                       cc.Variant.opt, 1, beta)
    place = lambda x, pinned: x.pin_memory() if pinned else x
    a, b = (place(torch.randn(2 * rows * K).half(), pinned_in) for rows in (M, N))
    c = place(torch.zeros(2 * M * N), pinned_c)
    pipe.RunHost(a.data_ptr(), b.data_ptr(), c.data_ptr())
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as trace:
        pipe.RunHost(a.data_ptr(), b.data_ptr(), c.data_ptr())
    names = [e.key for e in trace.key_averages()]
    fetched = any("copy_from_host" in n for n in names)
    copies = sum(e.count for e in trace.key_averages() if e.key == "hipMemcpyAsync")
    return int(fetched), copies

for case in [(1, 1, 64, 64, 64), (1, 0, 64, 64, 64), (0, 1, 64, 64, 64), (0, 0, 64, 64, 64), (1, 1, 64, 64, 64, 0.5),
             (1, 1, 64, 64, 20000), (1, 1, 1024, 1100, 40)]:
    print("route", case, *host_run(*case), flush=True)
"""


def test_route():
    """(In a process of its own: a profiler slows the launches that follow it.)"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(cc.__file__)))
    out = subprocess.run([sys.executable, "-c", PROGRAM], cwd=root, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    got = [line.split(") ")[1] for line in out.stdout.splitlines() if line.startswith("route")]
    assert got == [
        "1 0",   # page-locked: one kernel fetches the operands, the GEMM stores C
        "1 1",   # C copied back
        "0 2",   # A and B copied in
        "0 3",
        "1 1",   # beta: C fetched with the operands, and copied back
        "0 2",   # more than 4 MiB of operands
        "1 1",   # more than 8 MiB of C
    ], out.stdout
