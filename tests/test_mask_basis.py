"""Tile-13 passes in the basis of their own flip masks, where they are not
run one by one on a single register: the half-tile exchange emulated on the
host, the batched kernel, the two persistent forms; and the tile order of
registers of 2^14 tiles and more in the half-tile and persistent forms.
States equal the oracle's, or the plain kernel's, bit for bit."""

import ctypes as C
import math

import numpy as np
import pytest

from phase2_amd import _native as nat
from phase2_amd import synth
from test_pass_shape import _coset, _groups, _half_slot, _shape

TILE, LOW, DIMS = 13, 2, 11


def _masks(rng, n, extra=0):
    """11 masks, independent beyond the two low bits, and sums of them."""
    rank = nat.lib().ph2hip_span_rank
    while True:
        x = rng.integers(1, 1 << n, DIMS).astype(np.uint64)
        rot = (nat.Rot * DIMS)(*[nat.Rot(int(v), 0, 1.0, 0.0) for v in x])
        if rank(rot, C.c_size_t(DIMS), C.c_uint32(LOW)) == DIMS:
            break
    for _ in range(extra):
        i, j, at = rng.integers(0, len(x), 3)
        x = np.insert(x, at, x[i] ^ x[j])
    return x


def _in_mask_basis(x, groups):
    """Whether each of the 11 independent masks touches one gathered tile
    bit: groups of four terms then touch four, where dense masks in the
    echelon basis of their span touch nearly all."""
    rest = (1 << TILE) - (1 << LOW)
    for g in groups:
        touched = 0
        for u in g["u"]:
            touched |= u & rest
        if bin(touched).count("1") > 4:
            return False
    return True


@pytest.mark.parametrize("n,extra", [(15, 0), (20, 0), (28, 0), (15, 6),
                                     (20, 12), (33, 25)])
def test_exchange_emulated(n, extra):
    """Every exchange moves every amplitude of the tile to the slot where the
    next group looks for it, half by half."""
    rng = np.random.default_rng(n + extra)
    d, nthreads = 4, 1 << (TILE - 4)
    checked = 0
    for _ in range(2):
        x = _masks(rng, n, extra)
        z = rng.integers(0, 1 << n, len(x)).astype(np.uint64)
        rc, sh = _shape(x, z, TILE, LOW)
        assert rc == 0
        if not sh[3] & 4:
            continue
        gs = _groups(x, z, TILE, LOW)
        if extra == 0:
            assert _in_mask_basis(x, gs)
        for g0, g1 in zip(gs, gs[1:]):
            h, xk = g0["xh"], g0["xk"]
            assert g0["jpos"][xk] == h and g1["jpos"][xk] == h
            table = {}
            for j in range(nthreads):
                half = j >> xk & 1
                for w in range(1 << d):
                    v = _coset(g0, j, w, TILE, d)
                    assert v >> h & 1 == half
                    table[half, _half_slot(v, h, TILE)] = v
            assert len(table) == 1 << TILE
            for j in range(nthreads):
                for w in range(1 << d):
                    v = _coset(g1, j, w, TILE, d)
                    assert table[j >> xk & 1, _half_slot(v, h, TILE)] == v
            checked += 1
    assert checked > 0


class _Job(C.Structure):
    """struct ph2hip_batch_job."""
    _fields_ = [("amp_off", C.c_uint64), ("nqb", C.c_uint32),
                ("rot", C.POINTER(nat.Rot)), ("n", C.c_size_t),
                ("pass_len", C.POINTER(C.c_uint32)), ("npass", C.c_size_t)]


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [0, 1])
def test_batched_kernel(oracle, graph):
    """Three registers, three passes each in the half-tile form: direct
    launches, and the round graph."""
    nat.init()
    L = nat.lib()
    rng = np.random.default_rng(77)
    widths = (13, 16, 14)
    namp = sum(1 << n for n in widths)
    st = rng.normal(size=namp) + 1j * rng.normal(size=namp)
    want, jobs, keep, off = st.copy(), (_Job * 3)(), [], 0
    for i, n in enumerate(widths):
        xs = [_masks(rng, n) for _ in range(3)]
        for x in xs:
            assert _in_mask_basis(x, _groups(x, x, TILE, LOW))
            assert _shape(x, x, TILE, LOW)[1][3] & 4
        x = np.concatenate(xs)
        z = rng.integers(0, 1 << n, len(x)).astype(np.uint64)
        phi = rng.normal(size=len(x))
        rot = (nat.Rot * len(x))(*[
            nat.Rot(int(a), int(b), math.cos(p), math.sin(p))
            for a, b, p in zip(x, z, phi)])
        lens = (C.c_uint32 * 3)(*[len(v) for v in xs])
        jobs[i] = _Job(off, n, rot, len(x), lens, 3)
        keep += [rot, lens]
        want[off:off + (1 << n)] = oracle.rotate(st[off:off + (1 << n)], x, z,
                                                 phi)
        off += 1 << n
    amp = C.c_void_p()
    assert L.ph2hip_malloc(C.byref(amp), C.c_size_t(16 * namp)) == 0
    try:
        nat.prof_enable(not graph)
        nat.prof_records(reset=True)
        assert L.ph2hip_h2d(amp, st.ctypes.data_as(C.c_void_p),
                            C.c_size_t(16 * namp)) == 0
        nl = C.c_uint64(0)
        assert L.ph2hip_rotate_batched(
            amp, C.c_uint64(namp), jobs, C.c_size_t(3), C.c_uint32(TILE),
            C.c_uint32(LOW), C.c_int(graph), C.byref(nl)) == 0
        got = np.zeros(namp, complex)
        assert L.ph2hip_d2h(got.ctypes.data_as(C.c_void_p), amp,
                            C.c_size_t(16 * namp)) == 0
        rec = nat.prof_records(reset=True)
    finally:
        nat.prof_enable(False)
        L.ph2hip_free(amp)
    assert nl.value == 3
    if not graph:
        rec = rec[rec["kind"] == 3]
        assert len(rec) == 3 and np.all(rec["direct"] & 4)
    assert np.array_equal(got, want)


def _prefetch(tile, amps, wgs):
    assert nat.lib().ph2hip_set_fused_prefetch(
        C.c_uint32(tile), C.c_uint32(amps), C.c_uint32(wgs)) == 0


FORMS = {
    "half": (lambda t: None, lambda t: None),
    "prefetch8": (lambda t: _prefetch(t, 8, 2), lambda t: _prefetch(t, 0, 0)),
    "prefetch16": (lambda t: _prefetch(t, 16, 1),
                   lambda t: _prefetch(t, 0, 0)),
    "pipe": (lambda t: nat.set_fused_form(1 << t),
             lambda t: nat.set_fused_form(0)),
}


def _equals_plain(n, tile, name, x, z, phi):
    a, b = nat.Register(n, nat.FUSED, tile, LOW), nat.Register(n, nat.PLAIN)
    change, restore = FORMS[name]
    try:
        for r in (a, b):
            r.fill_hash(n)
        b.rotate(x, z, phi)
        change(tile)
        nat.prof_enable(True)
        nat.prof_records(reset=True)
        a.rotate(x, z, phi)
        rec = nat.prof_records(reset=True)
        nat.prof_enable(False)
        assert a.count_unequal(b) == 0
        return rec
    finally:
        nat.prof_enable(False)
        restore(tile)
        a.free()
        b.free()


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(FORMS))
@pytest.mark.parametrize("n", [13, 17, 22])
def test_forms_in_mask_basis(name, n):
    rng = np.random.default_rng(n)
    x = _masks(rng, n)
    assert _in_mask_basis(x, _groups(x, x, TILE, LOW))
    z = rng.integers(0, 1 << n, DIMS).astype(np.uint64)
    rec = _equals_plain(n, TILE, name, x, z, rng.normal(size=DIMS))
    assert len(rec) == 1 and rec["direct"][0] & 4


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(FORMS))
@pytest.mark.parametrize("n,tile", [(25, 12), (26, 12), (26, 13), (27, 13),
                                    (28, 13)])
def test_tile_order(name, n, tile):
    """Fewer than 2^14 tiles, exactly as many, and more."""
    hm = synth.hamiltonian(n, 300, seed=n)
    k = nat.sort_lex(hm.xm, hm.zm)[-200:-170]
    rec = _equals_plain(n, tile, name, hm.xm[k], hm.zm[k], hm.cf[k])
    assert set(rec["tile_bits"].tolist()) == {tile}
    assert np.any(rec["direct"] & 4)
