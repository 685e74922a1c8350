"""qreg_hip_device_ptr returns when everything queued on the register is done,
so that the buffer can be read on any stream: each time with a sweep of
another register still running on the library's stream, and a copy on the
null stream, which that stream does not order."""

import ctypes as C

import numpy as np
import pytest

from phase2_amd import _native as nat

pytestmark = pytest.mark.gpu

N = 12


@pytest.fixture(scope="module")
def busy():
    """Queues some milliseconds of sweeps on the library's stream."""
    rng = np.random.default_rng(1)
    reg = nat.Register(25)
    reg.fill_hash(1)
    x = rng.integers(0, 1 << 25, 200).astype(np.uint64)
    z = rng.integers(0, 1 << 25, 200).astype(np.uint64)
    phi = rng.normal(size=200)

    def queue():
        for _ in range(3):
            reg.rotate(x, z, phi)
    yield queue
    reg.free()


def _ptr(reg):
    L = nat.lib()
    L.qreg_hip_device_ptr.restype = C.c_void_p
    return L.qreg_hip_device_ptr(C.c_void_p(reg.h))


def _look(reg, ptr=None):
    L = nat.lib()
    got = np.zeros(1 << reg.nqb, complex)
    ptr = ptr or _ptr(reg)
    # the runtime that the library is linked with
    assert L.hipMemcpy(C.c_void_p(got.ctypes.data), C.c_void_p(ptr),
                       C.c_size_t(got.nbytes), C.c_int(2)) == 0
    return got


def _start(n):
    reg = nat.Register(n)
    reg.prep_multidet([3], [1.0])
    st = np.zeros(1 << n, complex)
    st[3] = 1.0
    assert np.array_equal(_look(reg), st)
    return reg, st


@pytest.mark.parametrize("n", [5, N])
@pytest.mark.parametrize("mode", [nat.FUSED, nat.PLAIN])
def test_after_rotations(oracle, busy, n, mode):
    rng = np.random.default_rng(n)
    reg, st = _start(n)
    reg.configure(mode, 0, 3)
    try:
        x = rng.integers(0, 1 << n, 20).astype(np.uint64)
        z = rng.integers(0, 1 << n, 20).astype(np.uint64)
        phi = rng.normal(size=20)
        for _ in range(4):              # the later ones replay a graph
            busy()
            reg.rotate(x, z, phi)
            st = oracle.rotate(st, x, z, phi)
            assert np.array_equal(_look(reg), st)
    finally:
        reg.free()


def test_after_zero_and_writes(busy):
    reg, _ = _start(N)
    L = nat.lib()
    L.qreg_zero.argtypes = [C.c_void_p]
    L.qreg_setamp.argtypes = [C.c_void_p, C.c_uint64, C.c_double, C.c_double]
    try:
        st = np.zeros(1 << N, complex)
        busy()
        L.qreg_zero(reg.h)
        assert np.array_equal(_look(reg), st)
        busy()
        L.qreg_setamp(reg.h, 9, 0.5, -0.5)
        st[9] = 0.5 - 0.5j
        assert np.array_equal(_look(reg), st)
    finally:
        reg.free()


def test_after_calls_of_the_library(busy):
    """A state that another call of the library writes: the hashed fill."""
    a, _ = _start(N)
    b = nat.Register(N)
    try:
        b.fill_hash(7)
        want = b.read()
        busy()
        a.fill_hash(7)
        assert np.array_equal(_look(a), want)
    finally:
        a.free()
        b.free()


@pytest.mark.parametrize("count", [1, 64, 65])
def test_error_check_waits_for_writes(busy, count):
    """qreg_error reports on writes that have landed: they are in the buffer
    when it returns, also the short ones that are sent without a wait."""
    reg, st = _start(N)
    L = nat.lib()
    L.qreg_setamp.argtypes = [C.c_void_p, C.c_uint64, C.c_double, C.c_double]
    L.qreg_error.argtypes = [C.c_void_p]
    L.qreg_error.restype = C.c_int
    try:
        ptr = _ptr(reg)
        busy()
        for i in range(count):
            L.qreg_setamp(reg.h, 10 + i, 0.25, float(i))
            st[10 + i] = 0.25 + 1j * i
        assert L.qreg_error(reg.h) == 0
        assert np.array_equal(_look(reg, ptr), st)
    finally:
        reg.free()
