"""A captured sweep is replayed under the kernel form it was captured in and
no other: after any setting of the form the same call launches the form asked
for, and the setting put back finds its graph again."""

import ctypes as C

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import synth

pytestmark = pytest.mark.gpu


def _prefetch(tile, amps, wgs):
    nat.lib().ph2hip_set_fused_prefetch(C.c_uint32(tile), C.c_uint32(amps),
                                        C.c_uint32(wgs))


# tile, setting, the setting put back
FORMS = {
    "direct": (11, lambda: nat.set_fused_direct(False),
               lambda: nat.set_fused_direct(True)),
    "half": (12, lambda: nat.set_fused_half(0),
             lambda: nat.set_fused_half(nat.HALF_TILES)),
    "pipe": (11, lambda: nat.set_fused_form(1 << 11),
             lambda: nat.set_fused_form(0)),
    "prefetch": (12, lambda: _prefetch(12, 8, 2),
                 lambda: _prefetch(12, 0, 0)),
}


@pytest.mark.parametrize("name", sorted(FORMS))
def test_replay_follows_the_form(oracle, name):
    tile, change, restore = FORMS[name]
    n = 15
    nat.init()
    L = nat.lib()
    L.ph2hip_replay_hits.restype = C.c_uint64
    hits = L.ph2hip_replay_hits
    assert L.ph2hip_set_replay(C.c_uint32(20)) == 0
    hm = synth.hamiltonian(n, 200, seed=9)
    phi = 0.1 * hm.cf / np.max(np.abs(hm.cf))
    st = np.zeros(1 << n, complex)
    st[5] = 1.0
    reg = nat.Register(n, nat.FUSED, tile, 3)
    try:
        reg.prep_multidet([5], [1.0])

        def step():
            nonlocal st
            h = int(hits())
            reg.rotate(hm.xm, hm.zm, phi)
            st = oracle.rotate(st, hm.xm, hm.zm, phi)
            return int(hits()) - h
        # remembered, captured, replayed; under the new form once more so
        assert [step() for _ in range(3)] == [0, 0, 1]
        change()
        assert [step() for _ in range(3)] == [0, 0, 1]
        restore()
        assert step() == 1
        assert np.array_equal(reg.read(), st)
    finally:
        restore()
        reg.free()
