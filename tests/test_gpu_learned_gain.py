"""The committed network's schedule against the library's own default, the
automatic greedy cut, on sweep blocks of a Hamiltonian it was not trained on
(generator seed 7).  Both are timed in turn, each round the other way, and
compared by their medians over all blocks.  At 26 qubits, the narrowest
registers it is installed for, it has to be the faster one; at 30, where the
two are even (single blocks from 0.974 to 1.013), it may lose no more than
3%."""

import ctypes as C
import time

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import costmodel as cm
from phase2_amd import synth

pytestmark = pytest.mark.gpu

_u32p = C.POINTER(C.c_uint32)


def _learned(reg, x, z, phi, sched):
    lens, tbs, lbs = (np.ascontiguousarray(a, np.uint32) for a in sched)
    L = nat.lib()
    L.ph2_reg_rotate_sched.restype = C.c_int
    assert L.ph2_reg_rotate_sched(
        C.c_void_p(reg.h), C.c_size_t(len(x)),
        x.ctypes.data_as(C.POINTER(C.c_uint64)),
        z.ctypes.data_as(C.POINTER(C.c_uint64)),
        phi.ctypes.data_as(C.POINTER(C.c_double)),
        lens.ctypes.data_as(_u32p), tbs.ctypes.data_as(_u32p),
        lbs.ctypes.data_as(_u32p), C.c_size_t(len(lens))) == 0


@pytest.mark.parametrize("n,picked,rounds,most", [(26, (2, 5, 8, 11), 7, 1.0),
                                                  (30, (2, 5, 8), 3, 1.03)])
def test_learned_against_the_automatic_cut(n, picked, rounds, most):
    nat.init()
    hm = synth.hamiltonian(n, 0, seed=7, decay=True, n_total=1024 * 14)
    k = nat.sort_lex(hm.xm, hm.zm)
    blocks = [tuple(np.ascontiguousarray(a[k][b * 1024:(b + 1) * 1024])
                    for a in (hm.xm, hm.zm, 0.02 * hm.cf)) for b in picked]
    reg = nat.Register(n, nat.FUSED, 0, 3)
    try:
        cm.install(cm.load()[0], min_qb=n)
        scheds = [cm.schedule(x, z, n) for x, z, _ in blocks]
        cm.uninstall()
        reg.fill_hash(n)
        t = np.zeros((2, len(blocks), rounds + 1))
        for r in range(rounds + 1):
            for i, b in enumerate(blocks):
                for w in (0, 1) if r % 2 else (1, 0):
                    nat.synchronize()
                    t0 = time.perf_counter()
                    if w:
                        _learned(reg, *b, scheds[i])
                    else:
                        reg.rotate(*b)
                    nat.synchronize()
                    t[w, i, r] = time.perf_counter() - t0
    finally:
        cm.uninstall()
        reg.free()
    auto, learned = np.median(t[:, :, 1:], axis=2).sum(axis=1)
    print(f"n={n}: automatic {auto * 1e3:.2f} ms, learned "
          f"{learned * 1e3:.2f} ms, gain {auto / learned:.4f}x")
    assert learned < most * auto
