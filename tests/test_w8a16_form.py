"""Which kernel an fp8 layer takes, on the CPU (the choice looks at sizes and at the
operands' alignment only)."""
import ctypes as C

import pytest

import pyc_amd

BASE = 1 << 40


def _form(M, N, K, x_off=0, w_off=0):
    f = pyc_amd.lib().pyc_hip_w8a16_form
    f.argtypes = [C.c_int] * 3 + [C.c_void_p] * 2
    return f(M, N, K, BASE + x_off, BASE + w_off)


@pytest.mark.parametrize("x_off,w_off", [(2, 0), (4, 0), (8, 0), (0, 1), (0, 4), (0, 8), (2, 3)])
def test_unaligned_operands_are_loaded_through_registers(x_off, w_off):
    """LDS-DMA (forms 1 to 5) moves 16-byte chunks from 16-byte boundaries: operands
    elsewhere take the token kernel or the split-K kernel that loads registers."""
    for M in (1, 2, 4, 5, 8, 16, 17, 32):
        for N, K in [(1024, 1040), (4096, 4112), (11008, 4096), (4096, 11008), (1024, 14336), (64, 16), (9, 1024)]:
            assert _form(M, N, K, x_off, w_off) in (0, 6)
            assert M > 4 or _form(M, N, K, x_off, w_off) == 0 or M * K * 2 > 60000


def test_aligned_operands():
    assert _form(1, 4096, 11008) == 0
    assert _form(32, 4096, 11008) == 1
    assert _form(32, 11008, 4096) == 3
    assert _form(32, 1024, 14336) == 5
    assert _form(32, 1024, 14352) == 6  # K no multiple of 128: items of 64 k
