"""The tile widths in bench.py's line are those of the passes that ran."""

import numpy as np
import pytest

import bench
from phase2_amd import _native
from phase2_amd import costmodel as cm
from phase2_amd import synth


def _rec(tiles, kind=2):
    r = np.zeros(len(tiles), dtype=_native.REC_DTYPE)
    r["kind"], r["tile_bits"], r["ms"], r["amps"] = kind, tiles, 1.0, 1.0
    return r


@pytest.mark.parametrize("tiles,want", [([10], 10), ([13, 12, 13], [12, 13]),
                                        ([9, 9], 9), ([], 0)])
def test_tiles_run(tiles, want):
    for kind in (2, 3):
        prof = {"fused": None, "batched": None}
        kernels = bench.dominant_fused(_rec(tiles, kind), prof, kind)[2]
        assert bench.tiles_run(kernels, 0) == want


@pytest.mark.gpu
@pytest.mark.parametrize("n,want", [(10, 10), (11, 10), (16, 10), (20, 11),
                                    (21, 11), (23, 13), (28, 13)])
def test_automatic_width_of_a_sweep(n, want):
    """A sweep of a few hundred terms under the automatic width, as a run of
    bench.py at that width reports it."""
    hm = synth.hamiltonian(n, 60 * n, seed=n)
    k = _native.sort_lex(hm.xm, hm.zm)[-600:]
    reg = _native.Register(n, _native.FUSED, 0, 3)
    try:
        reg.fill_hash(1)
        _native.prof_enable(True)
        _native.prof_records(reset=True)
        reg.rotate(hm.xm[k], hm.zm[k], hm.cf[k])
        rec = _native.prof_records(reset=True)
    finally:
        _native.prof_enable(False)
        reg.free()
    kernels = bench.dominant_fused(rec, {"fused": None})[2]
    assert bench.tiles_run(kernels, 0) == want
    if n == 23:
        # the width by the pass counts: 13 saves a twentieth or more
        p13, p12 = (len(cm.schedule(hm.xm[k], hm.zm[k], n, greedy=(t, 2))[0])
                    for t in (13, 12))
        assert 20 * p13 <= 19 * p12
