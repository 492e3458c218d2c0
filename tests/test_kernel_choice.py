"""Which kernel fp32 GEMM, LayerNorm and attention calls take, on the CPU (the choice looks at
sizes and at the operands' alignment only)."""
import ctypes as C

import pytest

import pyc_amd

BASE = 1 << 40


def _f32(bt, m, n, k, a_off=0, b_off=0):
    f = pyc_amd.lib().pyc_hip_gemm_f32_form
    f.argtypes = [C.c_int] * 4 + [C.c_void_p] * 2
    return f(int(bt), m, n, k, BASE + a_off, BASE + b_off)


@pytest.mark.parametrize("bt,m,n,k,staged", [
    (False, 3520, 7424, 320, True), (False, 1280, 1088, 320, True), (True, 384, 1536, 192, True),
    (True, 8320, 2176, 832, True), (True, 5504, 2112, 1664, True),
    (True, 1024, 1024, 2048, False), (False, 1024, 1024, 1024, False), (False, 4096, 4096, 4096, False)])
def test_f32_whole_tiles_off_16_bytes(bt, m, n, k, staged):
    """Whole tiles off a 16-byte boundary: the register-staged kernel where k is short,
    which takes them without guards; on 16-byte boundaries always the ring."""
    assert (_f32(bt, m, n, k, 4) == 0) == (_f32(bt, m, n, k, 0, 8) == 0) == staged
    assert _f32(bt, m, n, k) in (32, 64)


@pytest.mark.parametrize("bt,m,n,k,form", [
    (False, 1728, 2568, 64, 0), (False, 1465, 3792, 404, 0), (False, 2676, 560, 448, 64),
    (True, 3435, 2968, 664, 0), (True, 2805, 1600, 1400, 64), (False, 910, 1651, 144, 0),
    (False, 1472, 1980, 194, 64), (False, 700, 701, 702, 32), (True, 440, 440, 440, 32)])
def test_f32_ragged(bt, m, n, k, form):
    assert _f32(bt, m, n, k) == form


def test_f32_unusual_operands():
    assert _f32(True, 512, 512, 512, 1) == 0 and _f32(False, 512, 512, 512, 0, 2) == 0  # off 4 bytes
    assert _f32(True, 1 << 16, 64, 1 << 15) == 0                                        # 8 GiB of A


@pytest.mark.parametrize("dtype,rows,d,off,row", [
    (2, 14495, 61, 0, 0), (1, 27475, 91, 0, 0), (1, 100, 64, 2, 0), (1, 100, 65, 2, 1), (2, 2047, 192, 2, 1),
    (2, 2048, 192, 2, 0), (2, 2048, 193, 2, 1), (1, 1024, 504, 0, 0), (1, 1023, 504, 0, 1), (1, 5000, 520, 0, 1),
    (0, 5000, 64, 0, 0), (0, 5000, 68, 0, 1), (0, 5000, 63, 0, 0), (0, 50, 64, 0, 1),
    (1, 1, 3392, 0, 1), (1, 8000, 5003, 0, 1), (1, 1023, 4096, 0, 1), (1, 1024, 4096, 0, 0), (0, 3, 2, 0, 0),
    (1, 5, 7, 0, 0), (2, 3, 16400, 0, 0)])
def test_layernorm_row_kernel(dtype, rows, d, off, row):
    """Short rows, which the plain kernel reads with one to three loads per lane, stay
    with it (the row kernel took 1.1 to 1.8 times as long); long and few ones do not."""
    f = pyc_amd.lib().pyc_hip_layernorm_row_form
    f.argtypes = [C.c_int] * 3 + [C.c_void_p] * 4
    assert f(dtype, rows, d, BASE + off, BASE, BASE, BASE) == row


@pytest.mark.parametrize("bh,s,d,causal,form", [
    (63, 1126, 64, 0, 4), (16, 3300, 64, 0, 1), (66, 3064, 64, 0, 1), (32, 1000, 64, 0, 4),
    (256, 2048, 128, 1, 1), (32, 1196, 128, 1, 4), (8, 1260, 64, 1, 2), (32, 2551, 128, 0, 1)])
def test_attention_form(bh, s, d, causal, form):
    """The form that is the fastest of the three there, by more than a few percent where
    it is a small one."""
    f = pyc_amd.lib().pyc_hip_attention_form
    f.argtypes = [C.c_int] * 4
    assert f(bh, s, d, causal) == form
