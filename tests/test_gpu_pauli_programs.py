"""Planned Pauli sums (many terms in one pass) on the GPU: expectation values,
operators and time evolution against numpy / scipy, around the sizes of a
tile (2^12 amplitudes) and of a thread's share of it, with strings wider than
a tile, repeated terms, identities and complex coefficients."""
import math

import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.linalg import expm_multiply

pytestmark = pytest.mark.gpu

NMAT = {"X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]]}


def random_terms(n, count, weight, rng, complex_c=False):
    out = [([], 0.3)]
    for i in range(count):
        qs = rng.choice(n, size=int(rng.integers(1, min(weight, n) + 1)), replace=False)
        c = float(rng.normal()) + (1j * float(rng.normal()) if complex_c else 0)
        out.append(([(int(q), "XYZ"[int(rng.integers(3))]) for q in qs], c))
        if i % 6 == 5:
            out.append((out[-1][0], 0.25))
    out.append(([(q, "Y") for q in range(n)], 0.2))  # wider than a tile from 13 qubits on
    return out


def apply_sum(terms, psi):
    n = int(math.log2(len(psi)))
    i = np.arange(len(psi))
    out = np.zeros_like(psi)
    for term, c in terms:
        x = z = 0
        for q, p in term:
            x |= (p in "XY") << q
            z |= (p in "YZ") << q
        src = i ^ x
        sign = 1 - 2 * (np.array([bin(v).count("1") for v in range(1 << min(n, 8))])[src & z & 255] & 1)
        m = (src & z) >> 8
        while np.any(m):
            sign = sign * (1 - 2 * (m & 1))
            m = m >> 1
        out += c * (1j ** (bin(x & z).count("1") % 4)) * sign * psi[src]
    return out


def prepared(engine_mod, n, precision, seed):
    sim = engine_mod.SimulatorMPI(seed, n, 4, precision)
    sim.allocate_qureg(list(range(n)), 0)
    sim.init_random_state(seed)
    return sim


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [8, 9, 10, 11, 12, 13, 17])
def test_sums_match_numpy(engine_mod, n, precision):
    rng = np.random.default_rng(n)
    print("pauli sums n=%d %s" % (n, precision), flush=True)
    sim = prepared(engine_mod, n, precision, 5 + n)
    ids = list(range(n))
    psi = sim.get_state()
    eps = 2.0 ** -52 if precision == "c128" else 2.0 ** -23
    for terms in (random_terms(n, 40, 3, rng), random_terms(n, 12, n, rng, complex_c=True)):
        l1 = sum(abs(c) for _, c in terms)
        ref = np.vdot(psi, apply_sum(terms, psi))
        # FP64 sums of one addend a term and amplitude
        assert abs(sim.expectation_complex(terms, ids) - ref) <= 1e-13 * l1
        sim.snapshot()
        sim.apply_qubit_operator(terms, ids)
        got = sim.get_state()
        assert np.abs(got - apply_sum(terms, psi)).max() <= 4 * eps * len(terms) * l1 * np.abs(psi).max()
        sim.restore()


@pytest.mark.parametrize("n", [8, 9, 11, 12, 14])
def test_evolution_matches_expm(engine_mod, n):
    rng = np.random.default_rng(50 + n)
    terms = [t for t in random_terms(n, 20, 3, rng) if len(t[0]) <= 3]
    t = 0.37
    print("time evolution n=%d" % n, flush=True)
    mats = []
    for term, c in terms:
        m = sp.identity(1, format="csr")
        ops = dict(term)
        for q in reversed(range(n)):
            m = sp.kron(m, sp.csr_matrix(np.array(NMAT[ops[q]]) if q in ops else np.eye(2)), format="csr")
        mats.append(c * m)
    ham = sum(mats)
    for precision, tol in (("c128", 1e-10), ("c64", 2e-6)):
        sim = prepared(engine_mod, n, precision, 3)
        psi = sim.get_state()
        sim.emulate_time_evolution(terms, t, list(range(n)), [])
        ref = expm_multiply(-1j * t * ham, psi)
        assert np.abs(sim.get_state() - ref).max() <= tol, precision


@pytest.mark.parametrize("t,imag", [(-6.0, 0.0), (25.0, 0.0), (1e-9, 0.0), (0.4, 0.15)])
def test_evolution_long_backward_and_not_hermitian(engine_mod, t, imag):
    """Chebyshev series over long and negative times; a sum that is not Hermitian takes the Taylor steps."""
    n = 10
    terms = [([(i, "Z"), (i + 1, "Z")], 0.4 + 0.05 * i) for i in range(n - 1)] + [([(i, "X")], 0.3) for i in range(n)]
    if imag:
        terms.append(([(2, "Y"), (7, "X")], 1j * imag))
    mats = []
    for term, c in terms:
        m = sp.identity(1, format="csr")
        ops = dict(term)
        for q in reversed(range(n)):
            m = sp.kron(m, sp.csr_matrix(np.array(NMAT[ops[q]]) if q in ops else np.eye(2)), format="csr")
        mats.append(c * m)
    ham = sum(mats)
    print("time evolution t=%g imag=%g" % (t, imag), flush=True)
    sim = prepared(engine_mod, n, "c128", 3)
    psi = sim.get_state()
    sim.emulate_time_evolution(terms, t, list(range(n)), [])
    assert np.abs(sim.get_state() - expm_multiply(-1j * t * ham, psi)).max() <= 1e-10


def test_controlled_evolution_keeps_the_rest(engine_mod):
    n = 13
    rng = np.random.default_rng(4)
    terms = [([(a, "X"), (b, "Y")], float(rng.normal())) for a, b in [(0, 1), (5, 6), (2, 8)]] + [([(3, "Z")], 0.5)]
    ids = list(range(9))
    sim = prepared(engine_mod, n, "c128", 9)
    psi = sim.get_state()
    print("controlled evolution n=%d" % n, flush=True)
    sim.emulate_time_evolution(terms, 0.8, ids, [10, 12])
    got = sim.get_state()
    on = (np.arange(1 << n) >> 10 & 1) & (np.arange(1 << n) >> 12 & 1) == 1
    assert np.abs(got[~on] - psi[~on]).max() <= 1e-15
    sub = psi[on].reshape(4, 512)  # bits 9 and 11 select the rows
    mats = []
    for term, c in terms:
        m = sp.identity(1, format="csr")
        ops = dict(term)
        for q in reversed(range(9)):
            m = sp.kron(m, sp.csr_matrix(np.array(NMAT[ops[q]]) if q in ops else np.eye(2)), format="csr")
        mats.append(c * m)
    ref = expm_multiply(-0.8j * sum(mats), sub.T).T.reshape(-1)
    assert np.abs(got[on] - ref).max() <= 1e-10
