"""Workloads of the state-vector library and how to run one pass of each.

A case is a dict of plain values.  ``listed()`` names the standing cases,
``draw(rng)`` gives one more of the same ranges, ``prepare(case, seed)``
makes what a program holds before the call, ``run(state)`` makes one pass
through the public entry points, ``work(case)`` counts the bytes and FP64
operations the pass cannot do without and ``exact(case, seed)`` gives the
same outputs from plain torch in complex128.

Kinds:

``run``     ``phase2_amd.run``: Pauli strings, a basis state, one amplitude.
``trott``   first-order Trotter series from a multideterminant state.
``trott2``  second-order Trotter series from a Slater coefficient matrix.
``sweep``   one block of lexicographically ordered rotations (what a Trotter
            step hands to the register, at most 1024 terms) on a register
            that stays on the device; returns the register's amplitudes.
``qdrift``  qDRIFT samples of one register.
``cmpsit``  composite integrator samples of one register.
``batch``   qDRIFT samples of many registers of uneven width together.
"""

from __future__ import annotations

import itertools
import math

import numpy as np
import torch

import phase2_amd
from phase2_amd import _native, costmodel, synth

# Terms of a rotation cost 6 FP64 operations per amplitude: two products and
# one sum for each of its two components.
OPS = 6
BLOCK = 1024


def listed():
    return [
        # a two-orbital molecule (H2, four spin orbitals) from a script: the
        # time is the call itself
        dict(name="run_4q", kind="run", n=4, four=4),
        # a small active space from a script: a few hundred strings
        dict(name="run_12q", kind="run", n=12, four=220),
        # the 64-step series of the 16-qubit workload of bench.py, final
        # state read back
        dict(name="trott_16q", kind="trott", n=16, four=400, steps=64,
             ndet=1, read=True),
        # ten orbitals, six electrons, closed shell: a correlated start state
        # and its overlap in every second-order step
        dict(name="trott2_20q", kind="trott2", n=20, occ=3, four=1200,
             steps=3),
        # one block of a Trotter step on registers of 4 MiB to 32 GiB
        dict(name="sweep_18q", kind="sweep", n=18, terms=1024),
        dict(name="sweep_22q", kind="sweep", n=22, terms=1024),
        # the odd last block of a sweep
        dict(name="sweep_25q", kind="sweep", n=25, terms=611),
        # a handful of rotations, as a caller of the register API makes them
        dict(name="sweep_28q_short", kind="sweep", n=28, terms=9),
        # the large-register sweep under the learned schedule
        dict(name="sweep_31q", kind="sweep", n=31, terms=1024, learned=True),
        # random sequences, as the two samplers draw them
        dict(name="qdrift_20q", kind="qdrift", n=20, four=3000, samples=3,
             depth=400),
        dict(name="cmpsit_24q", kind="cmpsit", n=24, four=4000, samples=1,
             steps=2, length=300, depth=120),
        # an ensemble of small registers
        dict(name="batch_40", kind="batch", nreg=40, nmin=12, nmax=21,
             four=1500, samples=3, depth=300),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(
        rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["run", "trott", "trott2", "sweep", "sweep", "sweep",
                       "qdrift", "cmpsit", "batch"])
    if kind == "run":
        n = rng.randint(4, 14)
        return dict(kind=kind, n=n,
                    four=min(_log(rng, 2, 400), _most_four(n)))
    if kind == "trott":
        return dict(kind=kind, n=rng.randint(9, 19), four=_log(rng, 100, 1500),
                    steps=_log(rng, 1, 40), ndet=_log(rng, 1, 64),
                    read=rng.random() < 0.5)
    if kind == "trott2":
        sites = rng.randint(5, 11)
        return dict(kind=kind, n=2 * sites, occ=rng.randint(1, sites // 2),
                    four=_log(rng, 100, 1500), steps=_log(rng, 1, 6))
    if kind == "sweep":
        n = rng.randint(9, 30)
        return dict(kind=kind, n=n,
                    terms=min(_log(rng, 1, BLOCK), n + _most_four(n)),
                    learned=n >= 26 and rng.random() < 0.5)
    if kind == "qdrift":
        return dict(kind=kind, n=rng.randint(10, 23),
                    four=_log(rng, 400, 4000), samples=_log(rng, 1, 6),
                    depth=_log(rng, 40, 700))
    if kind == "cmpsit":
        return dict(kind=kind, n=rng.randint(12, 25),
                    four=_log(rng, 600, 4000), samples=rng.randint(1, 2),
                    steps=rng.randint(1, 3), length=_log(rng, 50, 400),
                    depth=_log(rng, 20, 300))
    nmin = rng.randint(9, 16)
    return dict(kind="batch", nreg=_log(rng, 2, 48), nmin=nmin,
                nmax=nmin + rng.randint(0, 6), four=_log(rng, 400, 3000),
                samples=rng.randint(1, 4), depth=_log(rng, 60, 500))


# -- inputs -------------------------------------------------------------------

def _most_four(n):
    return 2 * math.comb(n, 4)


def _hamil(n, four, seed):
    return synth.hamiltonian_vec(n, min(four, _most_four(n)), seed)


def _lex(xm, zm):
    """Order by the operators I < X < Y < Z from the top qubit down."""
    keys = []
    for x, z in zip(xm.tolist(), zm.tolist()):
        k = 0
        for q in range(max(x.bit_length(), z.bit_length()) - 1, -1, -1):
            zb = z >> q & 1
            k |= (2 * zb | (x >> q & 1) ^ zb) << (2 * q)
        keys.append(k)
    return np.array(sorted(range(len(keys)), key=keys.__getitem__),
                    dtype=np.int64)


def _dets(n, ndet, seed):
    return synth.multidet_random(n, min(ndet, math.comb(n, n // 2)), n // 2,
                                 seed)


def _strings(hm):
    out = []
    for x, z in zip(hm.xm.tolist(), hm.zm.tolist()):
        toks = []
        for q in range(hm.nqb):
            xb, zb = x >> q & 1, z >> q & 1
            if xb or zb:
                toks.append(("Z" if not xb else "Y" if zb else "X") + str(q))
        out.append(" ".join(toks) or "I0")
    return out


def _block(case, seed):
    """A run of consecutive terms of a lexicographic sweep and its angles."""
    n, terms = case["n"], case["terms"]
    fixed = n + n * (n - 1) // 2 + 1
    # a Hamiltonian of a few blocks to a few dozen, denser with the width
    four = max(terms, min(_most_four(n), 300 * n + 2 * terms))
    hm = _hamil(n, four, seed)
    terms = min(terms, len(hm))
    x, z, cf = hm.xm, hm.zm, hm.cf
    order = _lex(x, z)
    # sweeps begin with the diagonal terms; most blocks lie beyond them
    first = int(np.random.default_rng(seed).integers(
        0, len(hm) - terms + 1)) if len(hm) > fixed else 0
    pick = order[first:first + terms]
    return x[pick].copy(), z[pick].copy(), 0.2 * cf[pick]


def _occ_basis(n):
    return "".join("1" if q < n // 2 else "0" for q in range(n))


class _Amplitudes:
    """The register's device buffer, for torch to look at; keeps it alive."""

    def __init__(self, reg):
        ptr = _native.lib().qreg_hip_device_ptr
        ptr.restype = _native.C.c_void_p
        self.reg = reg
        self.__cuda_array_interface__ = dict(
            shape=(1 << reg.nqb, 2), typestr="<f8", version=2,
            data=(int(ptr(_native.C.c_void_p(reg.h))), False))


def _fill(t, n, seed):
    """A dense state, as a few Trotter steps leave it: complex Gaussian
    amplitudes, norm 1 within sampling error."""
    g = torch.Generator(device=t.device)
    g.manual_seed(seed)
    t.normal_(generator=g)
    t.mul_(2.0 ** (-(n + 1) / 2))


def prepare(case, seed):
    kind = case["kind"]
    _native.init()
    _native.set_default(_native.FUSED, 0, 3)
    if case.get("learned"):
        costmodel.install(costmodel.load()[0], 3, 26)
    else:
        costmodel.uninstall()
    if kind == "run":
        hm = _hamil(case["n"], case["four"], seed)
        return dict(kind=kind, paulis=_strings(hm), cf=hm.cf.tolist(),
                    psi=_occ_basis(case["n"]))
    if kind == "sweep":
        xm, zm, phi = _block(case, seed)
        reg = _native.Register(case["n"], _native.FUSED, 0, 3)
        amp = torch.as_tensor(_Amplitudes(reg), device="cuda")
        _fill(amp, case["n"], seed)
        torch.cuda.synchronize()
        return dict(kind=kind, reg=reg, amp=amp, xm=xm, zm=zm, phi=phi)
    if kind == "batch":
        return dict(kind=kind, regs=_registers(case, seed))
    hm = _hamil(case["n"], case["four"], seed)
    st = dict(kind=kind, hm=hm, case=case, seed=_stream_seed(seed))
    if kind == "trott2":
        c = synth.coeff_matrix(case["n"] // 2, case["occ"], seed)
        st["prep"] = dict(C_alpha=c, n_sites=case["n"] // 2,
                          n_alpha=case["occ"], n_beta=case["occ"],
                          closed_shell=1, tapered=0)
    else:
        idx, cf = _dets(case["n"], case.get("ndet", 4), seed)
        st["prep"] = dict(det_idx=idx, det_cf=cf)
    return st


def _stream_seed(seed):
    return 0x9E3779B97F4A7C15 ^ (seed + 1)


def _registers(case, seed):
    rng = np.random.default_rng(seed)
    regs = []
    for i in range(case["nreg"]):
        n = int(rng.integers(case["nmin"], case["nmax"] + 1))
        hm = _hamil(n, case["four"], 1000 * seed + i)
        idx, cf = _dets(n, 4, 1000 * seed + i)
        regs.append(dict(nqb=n, xm=hm.xm, zm=hm.zm, coeffs=hm.cf,
                         dets=dict(zip(idx.tolist(), cf.tolist())),
                         samples=case["samples"], depth=case["depth"],
                         step_size=0.01, seed=_stream_seed(1000 * seed + i)))
    return regs


# -- one pass -----------------------------------------------------------------

DELTA = 0.1
STEP = 0.05          # qDRIFT
ANGLE = 0.1          # composite integrator


def run(state):
    kind = state["kind"]
    if kind == "run":
        z = phase2_amd.run(state["paulis"], state["cf"], DELTA, state["psi"])
        return [z.real, z.imag]
    if kind == "sweep":
        state["reg"].rotate(state["xm"], state["zm"], state["phi"])
        return state["amp"]
    if kind == "batch":
        return phase2_amd.qdrift_batch(state["regs"])
    hm, prep, case = state["hm"], state["prep"], state["case"]
    if kind == "trott":
        ov, amp = _native.trott(1, hm, prep, DELTA, case["steps"],
                                want_state=case["read"])
        return [ov, amp] if case["read"] else [ov]
    if kind == "trott2":
        return [_native.trott(2, hm, prep, DELTA, case["steps"],
                              want_state=False)[0]]
    if kind == "qdrift":
        return [_native.qdrift(hm, prep, case["samples"], case["depth"], STEP,
                               state["seed"], want_state=False)[0]]
    return [_native.cmpsit(hm, prep, case["samples"], case["steps"],
                           case["length"], case["depth"], ANGLE, ANGLE / 50,
                           state["seed"], want_state=False)[0]]


# -- what a pass cannot do without --------------------------------------------

def _terms(case):
    n = case["n"]
    return n + n * (n - 1) // 2 + 1 + min(case["four"], _most_four(n))


def work(case):
    """The register once in and once out, the terms in, the results out."""
    kind = case["kind"]
    if kind == "batch":
        mean = sum(2.0 ** n for n in range(case["nmin"], case["nmax"] + 1)) \
            / (case["nmax"] + 1 - case["nmin"]) * case["nreg"]
        return dict(bytes=32 * mean * case["samples"],
                    flops=OPS * mean * case["samples"] * case["depth"])
    amps = 2.0 ** case["n"]
    if kind == "sweep":
        return dict(bytes=32 * amps + 24.0 * case["terms"],
                    flops=OPS * amps * case["terms"])
    passes, terms, out = 1, _terms(case), 1
    if kind == "trott":
        rot, out = terms * case["steps"], case["steps"]
        if case["read"]:
            out += amps
    elif kind == "trott2":
        rot, out = 2 * terms * case["steps"], case["steps"]
    elif kind == "qdrift":
        passes = out = case["samples"]
        rot = case["samples"] * case["depth"]
    elif kind == "cmpsit":
        passes = out = case["samples"]
        rot = 2 * case["samples"] * case["steps"] * (case["length"] +
                                                     case["depth"])
    else:
        rot = terms
    return dict(bytes=32 * amps * passes + 24.0 * terms + 16.0 * out,
                flops=OPS * amps * rot)


# -- the same in plain torch ---------------------------------------------------

def _parity(v):
    for s in (32, 16, 8, 4, 2, 1):
        v = v ^ (v >> s)
    return v & 1


class _Rotor:
    """exp(i phi P) on a complex128 state, for a fixed list of strings:
    P|j> = i^y (-1)^popcount(j & z) |j ^ x>, y = popcount(x & z)."""

    def __init__(self, n, xm, zm, dev):
        lo = n // 2
        hi = n - lo
        self.shape = (1 << hi, 1 << lo)
        x = torch.from_numpy(xm.astype(np.int64)).to(dev)[:, None]
        z = torch.from_numpy(zm.astype(np.int64)).to(dev)[:, None]
        r = torch.arange(1 << hi, device=dev)[None, :]
        c = torch.arange(1 << lo, device=dev)[None, :]
        self.row = r ^ (x >> lo)
        self.col = c ^ (x & ((1 << lo) - 1))
        self.srow = (1 - 2 * _parity(r & (z >> lo))).double()
        self.scol = (1 - 2 * _parity(c & z)).double()
        self.y = [bin(a & b).count("1") & 3
                  for a, b in zip(xm.tolist(), zm.tolist())]

    def apply(self, psi, k, phi):
        y = self.y[k]
        p = psi[self.row[k][:, None], self.col[k][None, :]]
        p.mul_(self.srow[k][:, None]).mul_(self.scol[k][None, :])
        f = 1j * math.sin(phi) * (1j ** y) * (-1) ** y
        return psi.mul_(math.cos(phi)).add_(p, alpha=f)


class _Xoshiro:
    """xoshiro256** seeded through splitmix64, the first 128 outputs left
    out; uniforms from the top 53 bits."""
    M = (1 << 64) - 1

    def __init__(self, seed):
        self.s = []
        for _ in range(4):
            seed = (seed + 0x9E3779B97F4A7C15) & self.M
            v = seed
            v = ((v ^ v >> 30) * 0xBF58476D1CE4E5B9) & self.M
            v = ((v ^ v >> 27) * 0x94D049BB133111EB) & self.M
            self.s.append(v ^ v >> 31)
        for _ in range(128):
            self.next()

    def _rotl(self, v, k):
        return (v << k | v >> (64 - k)) & self.M

    def next(self):
        s = self.s
        out = self._rotl(s[1] * 5 & self.M, 7) * 9 & self.M
        t = s[1] << 17 & self.M
        s[2] ^= s[0]
        s[3] ^= s[1]
        s[1] ^= s[2]
        s[0] ^= s[3]
        s[2] ^= t
        s[3] = self._rotl(s[3], 45)
        return out

    def draws(self, w, count):
        """Indices with probabilities |w|, by the cumulative table."""
        u = [(self.next() >> 11) * 2.0 ** -53 for _ in range(count)]
        w = np.abs(w)
        cdf = np.cumsum(w / np.cumsum(w)[-1])
        return np.minimum(np.searchsorted(cdf, u, side="right"), len(w) - 1)


def _start(rot, idx, cf, dev):
    psi = torch.zeros(rot.shape[0] * rot.shape[1], dtype=torch.complex128,
                      device=dev)
    psi[torch.from_numpy(idx.astype(np.int64)).to(dev)] = \
        torch.from_numpy(np.asarray(cf, np.complex128)).to(dev)
    return psi.view(rot.shape)


def _overlap(psi, idx, cf, dev):
    a = psi.reshape(-1)[torch.from_numpy(idx.astype(np.int64)).to(dev)]
    return complex(np.sum(a.cpu().numpy() * np.conj(cf)))


def _slater(c, occ):
    """Index and coefficient of every pair of alpha and beta occupations of
    a closed shell with orbitals ``c``."""
    sites = c.shape[0]
    subs = list(itertools.combinations(range(sites), occ))
    det = np.linalg.det(np.stack([c[list(s)] for s in subs]))
    mask = np.array([sum(1 << q for q in s) for s in subs], dtype=np.int64)
    cf = np.outer(det, det).reshape(-1)
    idx = (mask[:, None] | mask[None, :] << sites).reshape(-1)
    keep = np.abs(cf) >= 1e-12
    return idx[keep], cf[keep]


def _qdrift_exact(n, xm, zm, cf, idx, dcf, samples, depth, step, seed, dev):
    rot, rng, out = _Rotor(n, xm, zm, dev), _Xoshiro(seed), []
    omega = math.asin(step)
    for _ in range(samples):
        psi = _start(rot, idx, dcf, dev)
        for k in rng.draws(cf, depth).tolist():
            psi = rot.apply(psi, k, math.copysign(omega, cf[k]))
        out.append(_overlap(psi, idx, dcf, dev))
    return np.array(out)


def exact(case, seed):
    kind, dev = case["kind"], torch.device("cuda")
    w = work(case)
    # about 200 bytes of traffic per amplitude and rotation in plain torch
    if w["flops"] / OPS * 200 / 3e12 > 12:
        return None
    if kind == "batch":
        return [_qdrift_exact(
            r["nqb"], r["xm"], r["zm"], r["coeffs"],
            np.array(list(r["dets"]), dtype=np.int64),
            np.array(list(r["dets"].values())), r["samples"], r["depth"],
            r["step_size"], r["seed"], dev) for r in _registers(case, seed)]
    n = case["n"]
    if kind == "sweep":
        xm, zm, phi = _block(case, seed)
        t = torch.empty(1 << n, 2, dtype=torch.float64, device=dev)
        _fill(t, n, seed)
        rot = _Rotor(n, xm, zm, dev)
        psi = torch.view_as_complex(t).view(rot.shape)
        for k, a in enumerate(phi.tolist()):
            psi = rot.apply(psi, k, a)
        return torch.view_as_real(psi.reshape(-1))
    hm = _hamil(n, case["four"], seed)
    xm, zm, cf = hm.xm, hm.zm, hm.cf
    if kind == "run":
        rot = _Rotor(n, xm, zm, dev)
        idx = np.array([(1 << n // 2) - 1], dtype=np.int64)
        psi = _start(rot, idx, [1.0], dev)
        for k, a in enumerate(cf.tolist()):
            psi = rot.apply(psi, k, DELTA * a)
        z = _overlap(psi, idx, np.ones(1), dev)
        return [z.real, z.imag]
    if kind == "trott2":
        idx, dcf = _slater(synth.coeff_matrix(n // 2, case["occ"], seed),
                           case["occ"])
    else:
        idx, dcf = _dets(n, case.get("ndet", 4), seed)
    if kind == "qdrift":
        return [_qdrift_exact(n, xm, zm, cf, idx, dcf, case["samples"],
                              case["depth"], STEP, _stream_seed(seed), dev)]
    if kind == "cmpsit":
        order = np.argsort(-np.abs(cf), kind="stable")
        xm, zm, cf = xm[order], zm[order], cf[order]
        top = case["length"]
        lex = _lex(xm[:top], zm[:top]).tolist()
        rot, rng, out = _Rotor(n, xm, zm, dev), _Xoshiro(_stream_seed(seed)), []
        for _ in range(case["samples"]):
            psi = _start(rot, idx, dcf, dev)
            for half in range(2 * case["steps"]):
                ks = rng.draws(cf[top:], case["depth"]) + top
                seq = [(k, 0.5 * (cf[k] * ANGLE)) for k in lex] + \
                    [(k, 0.5 * math.copysign(ANGLE / 50, cf[k]))
                     for k in ks.tolist()]
                for k, a in reversed(seq) if half & 1 else seq:
                    psi = rot.apply(psi, k, a)
            out.append(_overlap(psi, idx, dcf, dev))
        return [np.array(out)]
    order = _lex(xm, zm)
    xm, zm, cf = xm[order], zm[order], cf[order]
    rot = _Rotor(n, xm, zm, dev)
    psi, out = _start(rot, idx, dcf, dev), []
    for _ in range(case["steps"]):
        if kind == "trott":
            seq = [(k, DELTA * a) for k, a in enumerate(cf.tolist())]
        else:
            seq = [(k, DELTA / 2 * a) for k, a in enumerate(cf.tolist())]
            seq += seq[::-1]
        for k, a in seq:
            psi = rot.apply(psi, k, a)
        out.append(_overlap(psi, idx, dcf, dev))
    if kind == "trott" and case["read"]:
        return [np.array(out), psi.reshape(-1).cpu().numpy()]
    return [np.array(out)]
