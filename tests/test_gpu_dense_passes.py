"""Tile-13 passes whose masks are dense: in the echelon basis of their span
most exchanges have no tile bit that both groups leave alone, so the pass
takes the basis of its own masks (and with it the half-tile form); tile
orders of registers of few and of many tiles; the cut without low bits that
narrow registers take for sweeps and not for random draws.  States equal the
oracle's bit for bit."""

import ctypes as C

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import synth


def _shape(xm, zm, tile, low):
    rot = (nat.Rot * len(xm))()
    for k in range(len(xm)):
        rot[k] = nat.Rot(int(xm[k]), int(zm[k]), 1.0, 0.0)
    sh = (C.c_uint32 * 4)()
    rc = nat.lib().ph2hip_pass_shape(rot, C.c_size_t(len(xm)),
                                     C.c_uint32(tile), C.c_uint32(low), sh)
    return rc, list(sh)


def _dense(rng, n, dims, extra):
    """dims masks that are independent beyond the two low bits, with extra
    sums of them, diagonal terms and repeats among them."""
    rank = nat.lib().ph2hip_span_rank
    while True:
        x = rng.integers(1, 1 << n, dims).astype(np.uint64)
        rot = (nat.Rot * dims)(*[nat.Rot(int(v), 0, 1.0, 0.0) for v in x])
        if rank(rot, C.c_size_t(dims), C.c_uint32(2)) == dims:
            break
    for _ in range(extra):
        i, j, at = rng.integers(0, len(x), 3)
        x = np.insert(x, at, x[i] ^ x[j] ^ np.uint64(rng.integers(0, 4)))
    return x, rng.integers(0, 1 << n, len(x)).astype(np.uint64)


@pytest.mark.parametrize("n", [15, 20, 28])
def test_dense_masks_keep_half_tile_form(n):
    rng = np.random.default_rng(n)
    half = sum(_shape(*_dense(rng, n, 11, 0), 13, 2)[1][3] >> 2 & 1
               for _ in range(50))
    assert half == 50


@pytest.mark.gpu
@pytest.mark.parametrize("n", [13, 14, 16, 19])
@pytest.mark.parametrize("extra", [0, 5, 30])
def test_dense_passes(oracle, n, extra):
    rng = np.random.default_rng(100 * n + extra)
    st = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    for dims in (5, 9, 11):
        x, z = _dense(rng, n, dims, extra)
        phi = rng.normal(size=len(x))
        want = oracle.rotate(st, x, z, phi)
        for low in (0, 2, 4):
            assert np.array_equal(
                nat.rotate(st, x, z, phi, nat.FUSED, 13, low), want), low


@pytest.mark.gpu
@pytest.mark.parametrize("n,tile", [(22, 9), (23, 9), (23, 10), (24, 10)])
def test_tile_order(n, tile):
    """Fewer than 2^14 tiles, exactly as many, and more."""
    rng = np.random.default_rng(n + tile)
    x = rng.integers(0, 1 << n, 40).astype(np.uint64)
    z = rng.integers(0, 1 << n, 40).astype(np.uint64)
    phi = rng.normal(size=40)
    a, b = nat.Register(n, nat.FUSED, tile, 2), nat.Register(n, nat.PLAIN)
    try:
        for r in (a, b):
            r.fill_hash(n)
            r.rotate(x, z, phi)
        assert a.count_unequal(b) == 0
    finally:
        a.free()
        b.free()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [10, 12, 13, 18, 19])
def test_automatic_low_bits(oracle, n):
    hm = synth.hamiltonian(n, 60 * n - 500 if n > 12 else 150, seed=n)
    lex = oracle.sort_lex(hm.xm, hm.zm)
    draw = np.random.default_rng(n).integers(0, len(hm.xm), 300)
    st = np.zeros(1 << n, complex)
    st[5] = 1.0
    reg = nat.Register(n, nat.FUSED, 0, 3)
    try:
        reg.prep_multidet([5], [1.0])
        low = []
        for k in (lex, draw, lex):
            phi = 0.1 * hm.cf[k] / np.max(np.abs(hm.cf))
            nat.prof_enable(True)
            nat.prof_records(reset=True)
            reg.rotate(hm.xm[k], hm.zm[k], phi)
            low.append(nat.prof_records(reset=True)["low_bits"].min())
            nat.prof_enable(False)
            st = oracle.rotate(st, hm.xm[k], hm.zm[k], phi)
        assert np.array_equal(reg.read(), st)
        assert low[0] == low[2]
        if n >= 19:
            assert min(low) >= 2
        if n in (13, 18):
            assert low[1] >= 2
    finally:
        nat.prof_enable(False)
        reg.free()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [21, 22, 24])
def test_automatic_tile(n):
    """A block of few terms at the width that costs its pass least, a sweep
    at the width that takes the fewest, without the half-tile form never 13;
    all equal to the plain sweep."""
    hm = synth.hamiltonian(n, 400, seed=n)
    lex = nat.sort_lex(hm.xm, hm.zm)
    a, b = nat.Register(n, nat.FUSED, 0, 3), nat.Register(n, nat.PLAIN)
    tiles = []
    try:
        for r in (a, b):
            r.fill_hash(n)
        for k, half in ((lex[300:304], nat.HALF_TILES),
                        (lex[200:], nat.HALF_TILES), (lex[200:], 0)):
            phi = 0.1 * hm.cf[k] / np.max(np.abs(hm.cf))
            nat.set_fused_half(half)
            nat.prof_enable(True)
            nat.prof_records(reset=True)
            a.rotate(hm.xm[k], hm.zm[k], phi)
            rec = nat.prof_records(reset=True)
            nat.prof_enable(False)
            tiles.append(set(rec["tile_bits"].tolist()))
            b.rotate(hm.xm[k], hm.zm[k], phi)
        assert a.count_unequal(b) == 0
        if n == 21:
            assert tiles == [{11}] * 3
        else:
            assert tiles[0] == {12} and tiles[2] == {12}
    finally:
        nat.prof_enable(False)
        nat.set_fused_half(nat.HALF_TILES)
        a.free()
        b.free()
