"""Contiguous low bits of the passes that the learned schedule chooses from:
three counts around the one asked for."""

import pytest

from phase2_amd import _native as nat
from phase2_amd import costmodel as cm
from phase2_amd import synth


@pytest.mark.parametrize("low,want", [(0, {0, 1, 2}), (1, {0, 1, 2}),
                                      (2, {1, 2, 3}), (3, {2, 3, 4}),
                                      (4, {3, 4, 5}), (7, {6, 7, 8})])
def test_candidate_low_bits(low, want):
    hm = synth.hamiltonian(28, 400, seed=3)
    k = nat.sort_lex(hm.xm, hm.zm)[-60:]
    cand = cm.candidates(hm.xm[k], hm.zm[k], 28, low)
    for tile in (12, 13):
        assert set(cand[cand[:, 2] == tile][:, 3].tolist()) == want


def test_default_is_the_middle_one():
    hm = synth.hamiltonian(28, 400, seed=3)
    k = nat.sort_lex(hm.xm, hm.zm)[-30:]
    a = cm.candidates(hm.xm[k], hm.zm[k], 28)
    assert (a == cm.candidates(hm.xm[k], hm.zm[k], 28, 3)).all()
