"""The half-GEMM dispatch on the CPU: hip_kernels.c is compiled with launchers
that record what they are asked for (and refuse what the real ones refuse), and
every accepted call has to compute each element of C exactly once."""
import ctypes as C
import os
import random
import subprocess

import pytest

import pyc_amd
from pyc_amd import build

RECORDER = r"""
#include <stddef.h>
typedef struct { int kind, bm, bn, m0, m1, n0, n1; } rec;  /* kind: 1 small, 2 nt, 3 nn, 4 register-staged */
static rec log_[16];
static int n_;
int rec_count(void) { return n_; }
const int* rec_get(int i) { return &log_[i].kind; }
void rec_clear(void) { n_ = 0; }
static int put(int kind, int bm, int bn, int m0, int m1, int n0, int n1) {
    log_[n_].kind = kind, log_[n_].bm = bm, log_[n_].bn = bn, log_[n_].m0 = m0, log_[n_].m1 = m1, log_[n_].n0 = n0;
    log_[n_++].n1 = n1;
    return 0;
}
int pyc_hip_gemm_small_takes(int, int, int, int, const void*, const void*);
int pyc_hip_gemm_nt_lds_takes(int, int, int, const void*, const void*, const void*, float, const float*, int);
int pyc_hip_gemm_nn_lds_takes(int, int, int, int, const void*, const void*, const void*, float, const float*, int);
int pyc_hip_gemm_half_launch(int bf, int bt, int tile, int M, int N, int K, const void* A, const void* B, void* C_,
                             float al, float be, const float* bias, int epi, void* s) {
    return put(4, tile, tile, 0, M, 0, N);
}
int pyc_hip_gemm_small_launch(int bf, int bt, int bm, int bn, int M, int N, int K, const void* A, const void* B,
                              void* C_, float al, float be, const float* bias, int epi, int m0, int m1, int n0, int n1,
                              void* s) {
    const int t = pyc_hip_gemm_small_takes(bt, M, N, K, A, B);
    if (t == 0 || (t == 1 && bn == 256) || m0 < 0 || m0 >= m1 || m1 > M || n0 < 0 || n0 >= n1 || n1 > N) return 1;
    return put(1, bm, bn, m0, m1, n0, n1);
}
int pyc_hip_gemm_nt_lds_launch(int bf, int M, int N, int K, const void* A, const void* B, void* C_, float al, float be,
                               const float* bias, int epi, int m_end, int n_end, void* s) {
    const int t = pyc_hip_gemm_nt_lds_takes(M, N, K, A, B, C_, be, bias, epi);
    return t ? put(2, t, 256, 0, m_end, 0, n_end) : 1;  /* bm: 1 one-shot, 2 persistent */
}
int pyc_hip_gemm_nn_lds_launch(int bf, int rag, int M, int N, int K, const void* A, const void* B, void* C_, float al,
                               float be, const float* bias, int epi, int m_end, int n_end, void* s) {
    return pyc_hip_gemm_nn_lds_takes(rag, M, N, K, A, B, C_, be, bias, epi) ? put(3, 2, 256, 0, m_end, 0, n_end) : 1;
}
int pyc_kernel_register(const void* d) { return 0; }
int pyc_kernel_promote_symbol(const char* a, int b, const char* c) { return 0; }
size_t pyc_kernel_collect(const char* a, int b, void* c, size_t n) { return 0; }
"""


@pytest.fixture(scope="module")
def dispatch(tmp_path_factory):
    d = tmp_path_factory.mktemp("dispatch")
    (d / "rec.c").write_text(RECORDER)
    so = d / "dispatch.so"
    host = os.path.join(build.HERE, "csrc", "host")
    pyc_amd.lib()
    subprocess.run(["gcc", "-shared", "-w", *[f for f in build.C_FLAGS if not f.startswith("-W")],
                    os.path.join(host, "hip_kernels.c"), str(d / "rec.c"), "-Wl,-Bsymbolic", build.LIB_PATH,
                    os.path.join(build.ROCM, "lib", "libamdhip64.so"), f"-Wl,-rpath,{build.LIB_DIR}", "-o", str(so)],
                   check=True)
    L = C.CDLL(str(so))
    L.rec_get.restype = C.POINTER(C.c_int)
    L.pyc_hip_gemm_dispatch.argtypes = ([C.c_char_p] + [C.c_int] * 3 + [C.c_void_p] * 3 + [C.c_float] * 2 +
                                        [C.c_void_p, C.c_int, C.c_void_p])
    L.pyc_hip_gemm_plan.argtypes = [C.c_int] * 4 + [C.c_void_p] * 3 + [C.c_float, C.c_void_p, C.c_int, C.c_void_p]
    return L


BASE = 1 << 40  # addresses are looked at for their alignment only


def _run(L, bt, m, n, k, a_off=0, b_off=0, c_off=0, bias_off=None, beta=0.0):
    L.rec_clear()
    bias = None if bias_off is None else BASE + bias_off
    rc = L.pyc_hip_gemm_dispatch(b"hip_gemm_bf16_nt" if bt else b"hip_gemm_bf16_nn", m, n, k, BASE + a_off, BASE + b_off,
                                 BASE + c_off, 1.0, beta, bias, 0 if bias is None else 1, None)
    return rc, [tuple(L.rec_get(i)[j] for j in range(7)) for i in range(L.rec_count())]


def _once(parts, m, n):
    """The parts' rectangles cover m x n once (they are one, or two that meet in a line)."""
    area = sum((p[4] - p[3]) * (p[6] - p[5]) for p in parts)
    if len(parts) == 2:
        a, b = parts
        assert (a[4] == b[3] and (a[5], a[6]) == (b[5], b[6]) == (0, n)) or \
               (a[6] == b[5] and (a[3], a[4]) == (b[3], b[4]) == (0, m)), parts
    assert 1 <= len(parts) <= 2 and area == m * n, parts


@pytest.mark.parametrize("bt", [True, False])
@pytest.mark.parametrize("m,n,k", [(4608, 4608, 1024), (4096, 6144, 4096)])
def test_part_that_is_refused_is_not_planned(dispatch, m, n, k, bt):
    """Operands off a 16-byte boundary at sizes whose aligned plan is 256 x 256 tiles
    and a rest of 128 x 256: the rest would be refused after the first part has run,
    and the product started again adds beta * C twice."""
    for a_off, b_off, beta in [(8, 0, 1.0), (0, 8, 1.0), (8, 8, 0.0), (2, 0, 0.5)]:
        rc, parts = _run(dispatch, bt, m, n, k, a_off, b_off, beta=beta)
        assert rc == 0
        _once(parts, m, n)


def test_every_call_computes_each_element_once(dispatch):
    rng = random.Random(7)
    split = 0
    for _ in range(4000):
        m, n, k = (max(1, int(2 ** rng.uniform(0, 13.5))) for _ in range(3))
        if rng.random() < 0.6:
            m, n, k = ((v + 63) // 64 * 64 for v in (m, n, k))
        elif rng.random() < 0.5:
            n, k = (n + 7) // 8 * 8, (k + 63) // 64 * 64
        off = lambda: rng.choice([0, 0, 0, 2, 4, 8])  # noqa: E731
        args = (rng.random() < 0.5, m, n, k, off(), off(), off(), rng.choice([None, 0, 4]), rng.choice([0.0, 0.0, 0.5]))
        rc, parts = _run(dispatch, *args)
        assert rc == 0, args
        _once(parts, m, n)
        split += len(parts) == 2
    assert split > 50


@pytest.mark.parametrize("m,n,k", [(3072, 4096, 2048), (3001, 4096, 1024), (1024, 4096, 4096)])
def test_one_shot_kernel_only_with_a_tile_per_cu(dispatch, m, n, k):
    """[N,K] products with beta, or with C off a 16-byte boundary, cannot take the
    persistent kernel; the one-shot kernel is slower than smaller tiles for them unless
    the 256 x 256 tiles fill the chip."""
    for kw in (dict(beta=0.5), dict(c_off=8), dict(c_off=8, bias_off=4)):
        rc, parts = _run(dispatch, True, m, n, k, **kw)
        assert rc == 0 and all(p[0] == 1 for p in parts), (kw, parts)
    rc, parts = _run(dispatch, True, 4096, 4096, k, beta=0.5)
    assert rc == 0 and parts[0][:2] == (2, 1)


@pytest.mark.parametrize("bt,m,n,k,off,general", [
    (False, 832, 768, 64, 2, True), (True, 3840, 3840, 64, 8, True), (True, 2048, 2048, 128, 8, True),
    (False, 64, 64, 64, 2, True), (True, 1, 330, 17, 0, True),
    (False, 5888, 1856, 320, 8, False), (False, 1280, 3072, 1600, 8, False), (True, 839, 7424, 2347, 0, False),
    (False, 3218, 922, 7424, 0, False)])
def test_short_k_off_16_bytes_takes_the_general_tiles(dispatch, bt, m, n, k, off, general):
    """Operands that LDS-DMA cannot move in whole chunks: the general tiles, which load
    them directly, are up to twice as fast as the register-staged ring at a short K,
    and far slower at a long one."""
    rc, parts = _run(dispatch, bt, m, n, k, off, off)
    assert rc == 0 and (parts[0][0] == 4) == general, parts
    rc, parts = _run(dispatch, bt, m, n, k)  # on 16-byte boundaries: as ever
    assert rc == 0 and (k % 8 != 0 or parts[0][0] != 4)
