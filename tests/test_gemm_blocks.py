"""Block shapes of the fp32 GEMM by rows, on the CPU (gemm_f32_config looks at
sizes only).  A launch takes about the time of the fullest CU's blocks, so a
larger block shape is right only where that CU gets no more work in it; and
each shape is picked somewhere in the range."""
import ctypes
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "boa-constrictor_amd")


class GemmArgs(ctypes.Structure):  # boa::GemmArgs (csrc/boa_kernels.h)
    _fields_ = [("X", ctypes.c_void_p), ("ldx", ctypes.c_int), ("W", ctypes.c_void_p),
                ("ldw", ctypes.c_int), ("C", ctypes.c_void_p), ("ldc", ctypes.c_int),
                ("bias", ctypes.c_void_p), ("res", ctypes.c_void_p), ("ldr", ctypes.c_int),
                ("M", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int), ("act", ctypes.c_int)]


@pytest.fixture(scope="module")
def config():
    f = getattr(ctypes.CDLL(os.path.join(PKG, "libboa_hip.so")),
                "_ZN3boa15gemm_f32_configERKNS_8GemmArgsE")
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.POINTER(GemmArgs)]
    return lambda m, n, k: f(ctypes.byref(GemmArgs(M=m, N=n, K=k)))


@pytest.mark.parametrize("d", [64, 80, 128, 256, 512])
def test_no_more_work_on_the_fullest_cu(config, d):
    def blocks(bm, bn):
        return -(-(-(-m // bm) * -(-n // bn)) // 256)

    picked = set()
    shapes = [(4 * d, d), (d, 2 * d), (d, 4 * d), (d, d), (256, d), (48, 2 * d), (96, 2 * d)]
    for n, k in shapes:
        for m in range(1, 16384, 61):
            c = config(m, n, k)
            picked.add(c)
            # work in units of a 32 x 32 block
            work = {1: 8 * blocks(128, 64), 2: blocks(32, 32), 3: 2 * blocks(64, 32)}[c]
            # (measured, a unit in a 128 x 64 block takes 10 to 17 % less)
            assert work <= blocks(32, 32) * (8 / 7 if c == 1 else 1), (m, n, k, c)
            assert c != 3 or k % 32 == 0
    assert picked == ({1, 2, 3} if d > 128 else {2, 3} if d == 128 else {2})
