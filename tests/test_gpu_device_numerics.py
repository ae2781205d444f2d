"""The device arithmetic that replaces longer forms (tests/device_numerics.hip),
over every float: the reciprocal against the division, the UNORM8 pack against
clamp, scale and round per channel, the fraction and the clamped 16-bit
coordinate against their ordered selects."""
import ctypes
import os

import pytest
import torch

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libswr_numerics.so")


def test_every_float():
    assert os.path.exists(LIB), "tests/libswr_numerics.so is not built (python __graft_entry__.py)"
    lib = ctypes.CDLL(LIB)
    lib.swr_numerics_sweep.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    bad = torch.zeros(4, dtype=torch.int64, device="cuda:0")
    arg = torch.zeros(4, dtype=torch.int32, device="cuda:0")
    torch.cuda.synchronize()
    print("[device numerics] 2^32 arguments", flush=True)
    assert lib.swr_numerics_sweep(bad.data_ptr(), arg.data_ptr()) == 0
    torch.cuda.synchronize()
    names = ("reciprocal", "UNORM8 pack", "fraction", "clamped 16-bit coordinate")
    wrong = {n: (b, hex(a & 0xFFFFFFFF)) for n, b, a in zip(names, bad.tolist(), arg.tolist()) if b}
    assert not wrong, wrong
