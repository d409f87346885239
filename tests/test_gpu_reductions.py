"""Probabilities, entropy, collapse, measurement, deallocation and Pauli
expectation values on the GPU against numpy, around the sizes where their
kernels change form: one block (2^8 amplitudes), the single-workgroup removal
of a qubit (2^12), the largest grid and its unrolled loop (2^18, 2^21), the
removal without a wait (2^20), and lists of strings around one launch's
eight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def prepared(engine_mod, n, precision, seed):
    rng = np.random.default_rng(seed)
    wf = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    wf /= np.linalg.norm(wf)
    sim = engine_mod.SimulatorMPI(seed, n, 4, precision)
    sim.allocate_qureg(list(range(n)), 0)
    sim.set_wavefunction(wf, list(range(n)))
    return sim, wf.astype(np.complex64).astype(np.complex128) if precision == "c64" else wf


def eps(n, precision, amplitudes=False):
    """Sums of 2^n terms in FP64, in any order; amplitudes that were scaled are rounded to the precision."""
    return 2.0 ** (n - 51) + (0 if not amplitudes else (2.0 ** -22 if precision == "c64" else 2.0 ** -50))


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 18, 19, 21, 22])
def test_probability_entropy_collapse(engine_mod, n, precision):
    sim, psi = prepared(engine_mod, n, precision, 20 + n)
    print("reductions n=%d %s" % (n, precision), flush=True)
    p = np.abs(psi) ** 2
    i = np.arange(1 << n)
    for ask in ([0], [n - 1], [0, n - 1], [n // 2, n - 1]):
        ask = list(dict.fromkeys(ask))
        ref = p[np.all([(i >> q) & 1 == 1 for q in ask], axis=0)].sum()
        assert abs(sim.get_probability([True] * len(ask), ask) - ref) <= eps(n, precision)
    ref = -(p * np.log2(p)).sum()
    assert abs(sim.entropy() - ref) <= eps(n, precision) * 4 * (n + 8)
    q = n // 2
    sim.collapse_wavefunction([q], [True])
    kept = np.where((i >> q) & 1, psi, 0)
    kept /= np.linalg.norm(kept)
    got = np.asarray(sim.get_state())
    assert np.all(got[((i >> q) & 1) == 0] == 0)
    assert np.abs(got - kept).max() <= eps(n, precision, True)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 6, 11, 12, 13, 20, 21])
def test_measure_then_deallocate(engine_mod, n, precision):
    sim, psi = prepared(engine_mod, n, precision, 40 + n)
    print("measure and deallocate n=%d %s" % (n, precision), flush=True)
    left = list(range(n))
    for q in dict.fromkeys([0, n - 1, n // 2]):
        if n > 1:
            with pytest.raises(RuntimeError, match="entangled"):
                sim.deallocate_qubit(q)
        (bit,) = sim.measure_qubits([q])
        at = left.index(q)
        i = np.arange(len(psi))
        kept = psi[((i >> at) & 1) == int(bit)]
        psi = kept / np.linalg.norm(kept)
        sim.deallocate_qubit(q)
        left.remove(q)
        got = np.asarray(sim.get_state())
        assert got.shape == psi.shape
        assert np.abs(got - psi).max() <= 3 * eps(n, precision, True)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n,terms", [(1, 1), (4, 7), (8, 8), (8, 9), (8, 17), (14, 9)])
def test_lists_of_strings(engine_mod, n, terms, precision):
    """Below 9 qubits, or with x parts wider than a tile of 12 bits, the strings go in lists of eight."""
    sim, psi = prepared(engine_mod, n, precision, 60 + n)
    print("strings n=%d terms=%d %s" % (n, terms, precision), flush=True)
    rng = np.random.default_rng(terms)
    mats = {"X": np.array([[0, 1], [1, 0]]), "Y": np.array([[0, -1j], [1j, 0]]), "Z": np.diag([1, -1])}
    total, spec = 0.0, []
    for _ in range(terms):
        ops = "".join(rng.choice(list("XY" if n > 12 else "XYZ"), size=n))
        c = float(rng.normal())
        v = psi
        for q in range(n):
            v = np.moveaxis(np.tensordot(mats[ops[q]], v.reshape((2,) * n), axes=([1], [n - 1 - q])), 0, n - 1 - q).reshape(-1)
        total += c * np.vdot(psi, v).real
        spec.append(([(q, ops[q]) for q in range(n)], c))
    got = sim.get_expectation_value(spec, list(range(n)))
    assert abs(got - total) <= terms * 8 * (eps(n, precision) + 2.0 ** -48)


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [0, 1, 9, 10, 11, 15, 16, 17, 18])
def test_state_comes_back(engine_mod, n, precision):
    """One workgroup up to 2^10 amplitudes, chunks of 2^16 in two buffers above."""
    print("readback n=%d %s" % (n, precision), flush=True)
    if n == 0:
        assert np.array_equal(engine_mod.SimulatorMPI(1, 4, 4, precision).get_state(), [1.0])
        return
    sim, psi = prepared(engine_mod, n, precision, 80 + n)
    assert np.array_equal(sim.get_state(), psi)
    assert np.array_equal(sim.get_state(), psi)
