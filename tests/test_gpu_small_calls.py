"""Short calls at the sizes where their path changes: amplitudes set by
kernel arguments (up to 64), through pinned memory (up to 8192) and through
device buffers, repeated indices, gathers of the same sizes, the first and
the second single read after a change, blocks that a register has seen
before, more blocks than it keeps, settings changed between two uses of a
block, and the batch tuner with registers narrower than its tiles.  Every
comparison is exact."""

import ctypes as C

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import synth

pytestmark = pytest.mark.gpu

N = 14


@pytest.mark.parametrize("count", [1, 64, 65, 8192, 8193])
def test_set_and_gather(count):
    rng = np.random.default_rng(count)
    idx = rng.integers(0, 1 << N, count).astype(np.uint64)
    idx[count // 2:count // 2 + 3] = idx[0]      # the last entry wins
    cf = rng.normal(size=count) + 1j * rng.normal(size=count)
    want = np.zeros(1 << N, complex)
    for i, z in zip(idx, cf):
        want[i] = z
    reg = nat.Register(N)
    try:
        reg.prep_multidet(idx, cf)
        assert np.array_equal(reg.gather(idx), want[idx.astype(int)])
        assert np.array_equal(reg.read(), want)
    finally:
        reg.free()


@pytest.mark.parametrize("count", [64, 65])
def test_set_on_another_stream(count):
    """The pointer is good for any stream once it is returned: a copy on the
    null stream, which the library's own stream does not order."""
    rng = np.random.default_rng(count)
    idx = rng.permutation(1 << N)[:count].astype(np.uint64)
    cf = rng.normal(size=count) + 1j * rng.normal(size=count)
    want = np.zeros(1 << N, complex)
    want[idx.astype(int)] = cf
    reg = nat.Register(N)
    try:
        L = nat.lib()
        L.qreg_hip_device_ptr.restype = C.c_void_p
        hip = C.CDLL("libamdhip64.so.7")
        got = np.zeros(1 << N, complex)
        reg.prep_multidet(idx, cf)
        ptr = L.qreg_hip_device_ptr(C.c_void_p(reg.h))
        assert hip.hipMemcpy(C.c_void_p(got.ctypes.data), C.c_void_p(ptr),
                             C.c_size_t(got.nbytes), C.c_int(2)) == 0
        assert np.array_equal(got, want)
    finally:
        reg.free()


def _block(rng, n, count):
    return (rng.integers(0, 1 << n, count).astype(np.uint64),
            rng.integers(0, 1 << n, count).astype(np.uint64),
            rng.normal(size=count))


@pytest.mark.parametrize("n", [7, 11, 15])
def test_blocks_kept(oracle, n):
    """11 blocks in turn (8 are kept), the same codes with other angles, and
    a change of tile, low bits, mode and half-tile form between uses."""
    rng = np.random.default_rng(n)
    blocks = [_block(rng, n, c) for c in (1, 5, 40, 40, 3, 90, 7, 7, 2, 60, 33)]
    x, z, p = blocks[2]
    blocks.insert(3, (x, z, -p))
    st = np.zeros(1 << n, complex)
    st[3] = 1.0
    reg = nat.Register(n)
    try:
        reg.prep_multidet([3], [1.0])
        for rep, (mode, tile, low, half) in enumerate([
                (nat.FUSED, 0, 3, nat.HALF_TILES), (nat.FUSED, 0, 3, 0),
                (nat.FUSED, 13, 3, nat.HALF_TILES), (nat.FUSED, 13, 3, 0),
                (nat.FUSED, 10, 2, nat.HALF_TILES),
                (nat.PLAIN, 0, 3, nat.HALF_TILES)]):
            if tile > n:
                tile = 0
            reg.configure(mode, tile, low)
            nat.set_fused_half(half)
            order = range(len(blocks)) if rep % 2 else [2, 3, 2, 3, 0, 1, 2]
            for b in order:
                x, z, p = blocks[b]
                reg.rotate(x, z, p)
                st = oracle.rotate(st, x, z, p)
            assert np.array_equal(reg.read(), st), rep
    finally:
        nat.set_fused_half(nat.HALF_TILES)
        reg.free()


def test_single_reads(oracle):
    """A read after a change takes the amplitude alone, the next ones a
    window; both see every write and rotation before them."""
    rng = np.random.default_rng(5)
    reg = nat.Register(N)
    L = nat.lib()
    L.qreg_getamp.argtypes = [C.c_void_p, C.c_uint64, C.POINTER(C.c_double)]
    L.qreg_setamp.argtypes = [C.c_void_p, C.c_uint64, C.c_double, C.c_double]
    z = (C.c_double * 2)()

    def get(i):
        L.qreg_getamp(reg.h, int(i), z)
        return complex(z[0], z[1])
    try:
        reg.prep_multidet([1], [1.0])
        st = np.zeros(1 << N, complex)
        st[1] = 1.0
        for k in range(3):
            b = _block(rng, N, 50)
            reg.rotate(*b)
            st = oracle.rotate(st, *b)
            for i in (7, 7, 8, 9)[k:]:
                assert get(i) == st[i]
                L.qreg_setamp(reg.h, i + 1, 0.5, -0.25 * k)
                st[i + 1] = complex(0.5, -0.25 * k)
                assert get(i + 1) == st[i + 1]
                assert get(i) == st[i]
        assert np.array_equal(reg.read(), st)
    finally:
        reg.free()


@pytest.mark.parametrize("widths", [[3], [6, 8], [9, 12], [10, 10, 13],
                                    [11, 12], [13, 14], [5, 9, 13]])
def test_batch_tuner(oracle, widths):
    regs = []
    for i, n in enumerate(widths):
        rng = np.random.default_rng(20 + i)
        x, z, c = _block(rng, n, 6 * n)
        hm = synth.Hamiltonian(n, x, z, c / np.sum(np.abs(c)))
        idx, cf = synth.multidet_random(n, 2, n // 2, seed=40 + i)
        regs.append(dict(hm=hm, det_idx=idx, det_cf=cf, samples=1 + i,
                         depth=60, step_size=0.03, seed=0x51 + i))
    got, st = nat.batch_qdrift(regs, nat.BATCH_FUSED_BATCHED, 0, 3)
    assert 9 <= st["tile_bits"] <= 13 and 2 <= st["low_bits"] <= 4
    for r, g in zip(regs, got):
        want, _ = oracle.qdrift(r["hm"], dict(det_idx=r["det_idx"],
                                              det_cf=r["det_cf"]),
                                r["samples"], r["depth"], r["step_size"],
                                r["seed"], want_state=False)
        assert np.array_equal(g, want)
