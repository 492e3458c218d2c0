"""The convolution's split of k into (tap row, tap column, channel) by rounded-up
reciprocals, on the CPU: exact for every k of every filter that is accepted, and
the filters for which it is not are refused (the general kernels, which divide, take
them)."""
import ctypes as C

import numpy as np
import pytest

import pyc_amd


def _split(R, S, Cin):
    rc, rs = C.c_uint32(), C.c_uint32()
    f = pyc_amd.lib().pyc_hip_conv2d_tap_split
    f.argtypes = [C.c_int] * 3 + [C.c_void_p] * 2
    return f(R, S, Cin, C.byref(rc), C.byref(rs)), rc.value, rs.value


def _exact(R, S, Cin, rc, rs):
    """What the kernel computes, for the first and last k of every tap."""
    t = np.arange(R * S, dtype=np.uint64)
    ok = True
    for k in (t * np.uint64(Cin), t * np.uint64(Cin) + np.uint64(Cin - 1)):
        ok &= bool(((k * np.uint64(rc)) >> np.uint64(32) == t).all())
    r = (t * np.uint64(rs)) >> np.uint64(32) if rs else t
    return ok and bool((r == t // np.uint64(S)).all())


@pytest.mark.parametrize("R,S,Cin", [(1, 65537, 8), (1649, 1649, 8), (3, 100003, 8), (46341, 1291, 8)])
def test_filters_the_split_gets_wrong_are_refused(R, S, Cin):
    ok, rc, rs = _split(R, S, Cin)
    assert not ok and not _exact(R, S, Cin, rc, rs)


def test_accepted_splits_are_exact():
    r = np.random.default_rng(3)
    shapes = [(1, 1, 8), (3, 3, 2048), (7, 7, 24), (1, 65536, 8), (2, 65535, 8), (5, 3, 8192), (255, 257, 8)]
    for _ in range(1500):
        shapes.append((int(2 ** r.uniform(0, 9)), int(2 ** r.uniform(0, 14)), 8 * int(2 ** r.uniform(0, 10))))
    taken = 0
    for R, S, Cin in shapes:
        ok, rc, rs = _split(R, S, Cin)
        if ok:
            taken += 1
            assert _exact(R, S, Cin, rc, rs), (R, S, Cin)
    assert taken > 500
    for R in (1, 2, 3, 5, 7, 11):     # ordinary filters stay accepted
        for S in (1, 2, 3, 5, 7, 11):
            for Cin in (8, 24, 64, 192, 1000, 2048):
                assert _split(R, S, Cin)[0]
