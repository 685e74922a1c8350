"""Fused passes at the edges of their descriptors: every tile width, one to a
few tiles, one term and the most terms, one micro-group and one per term,
diagonal and identity terms, first and last groups that move straight between
HBM and registers or through LDS.  The state equals the oracle's bit for bit
(the contract: every result is round(round(c u) +- round(s v)))."""

import numpy as np
import pytest

from phase2_amd import _native as nat

pytestmark = pytest.mark.gpu


def _terms(rng, n, count, kind):
    if kind == "one":          # one flipped qubit: one micro-group
        xm = np.full(count, 1 << (n - 1), dtype=np.uint64)
    elif kind == "each":       # no two consecutive flips share a qubit pair
        q = np.arange(count)
        xm = (np.uint64(1) << (q % n).astype(np.uint64)) | \
            (np.uint64(1) << ((5 * q + 3) % n).astype(np.uint64))
    else:                      # dense masks, diagonal and identity terms
        xm = rng.integers(0, 1 << n, count).astype(np.uint64)
        xm[::5] = 0
    zm = rng.integers(0, 1 << n, count).astype(np.uint64)
    zm[::7] = 0
    return xm, zm, rng.normal(size=count)


@pytest.mark.parametrize("tile", [9, 10, 11, 12, 13])
@pytest.mark.parametrize("extra", [0, 1, 3])
@pytest.mark.parametrize("kind", ["one", "each", "dense"])
def test_pass_edges(oracle, tile, extra, kind):
    n = tile + extra
    rng = np.random.default_rng(100 * tile + 10 * extra + len(kind))
    st = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    st[:4] = [0.0, -0.0, 1e-310, 1e300]      # zeros, a denormal, a large one
    for count in (1, 48, 97):
        xm, zm, phi = _terms(rng, n, count, kind)
        want = oracle.rotate(st, xm, zm, phi)
        for low in (0, 3, 5):
            for direct in (True, False):
                nat.set_fused_direct(direct)
                try:
                    got = nat.rotate(st, xm, zm, phi, nat.FUSED, tile, low)
                finally:
                    nat.set_fused_direct(True)
                assert np.array_equal(got, want), (count, low, direct)
