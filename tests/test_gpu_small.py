"""Registers of 1 to 8 qubits (ph2hip_rotate_small): runs that end at, before
and after the terms of one launch, diagonal, identity and dense masks; equal
to the oracle bit for bit."""

import numpy as np
import pytest

from phase2_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 5, 7, 8])
@pytest.mark.parametrize("count", [1, 127, 128, 129, 300])
def test_small_register(oracle, n, count):
    rng = np.random.default_rng(10 * n + count)
    st = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    st[0] = -0.0
    xm = rng.integers(0, 1 << n, count).astype(np.uint64)
    xm[::4] = 0
    zm = rng.integers(0, 1 << n, count).astype(np.uint64)
    zm[::5] = 0
    phi = rng.normal(size=count)
    want = oracle.rotate(st, xm, zm, phi)
    assert np.array_equal(nat.rotate(st, xm, zm, phi, nat.FUSED, 0, 3), want)
    assert np.array_equal(nat.rotate(st, xm, zm, phi, nat.PLAIN), want)
