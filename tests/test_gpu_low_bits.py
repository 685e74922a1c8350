"""Contiguous low bits that a caller sets are the ones its blocks are cut
with, also where the tile width is automatic: the passes that ran are those
of the greedy cut at the same tile and low bits.  Only the default (3) leaves
them to the library there."""

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import costmodel as cm
from phase2_amd import synth

pytestmark = pytest.mark.gpu

TILE = {11: 10, 14: 10, 18: 10, 19: 11, 21: 11, 28: 13}


def _ran(reg, x, z, phi):
    """(terms of every pass, tile width) of one sweep."""
    nat.prof_enable(True)
    nat.prof_records(reset=True)
    try:
        reg.rotate(x, z, phi)
        rec = nat.prof_records(reset=True)
    finally:
        nat.prof_enable(False)
    assert set(rec["tile_bits"].tolist()) == {TILE[reg.nqb]}
    return rec["nterms"].tolist()


@pytest.mark.parametrize("n", sorted(TILE))
def test_asked_for_low_bits(n):
    hm = synth.hamiltonian(n, 60 * n - 500, seed=n)
    lex = nat.sort_lex(hm.xm, hm.zm)[-250:]
    draw = np.random.default_rng(n).integers(0, len(hm.xm), 120)
    reg = nat.Register(n, nat.FUSED, 0, 3)
    try:
        reg.fill_hash(n)
        for k in (lex, draw):
            x, z = hm.xm[k], hm.zm[k]
            cut = {low: cm.schedule(x, z, n, greedy=(TILE[n], low))[0].tolist()
                   for low in range(6)}
            assert len(set(map(tuple, cut.values()))) > 1
            for low in (4, 5, 2, 1, 0):
                reg.configure(nat.FUSED, 0, low)
                assert _ran(reg, x, z, hm.cf[k]) == cut[low], low
            reg.configure(nat.FUSED, 0, 3)
            assert _ran(reg, x, z, hm.cf[k]) in (cut[2], cut[0])
    finally:
        reg.free()
