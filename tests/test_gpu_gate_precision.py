"""Long complex64 gate lists against the same lists in complex128.

Lists held in FP64 (the same angles again and again, many rotations a qubit, long runs on few
qubits) round each amplitude once a pass, by 2^-24 of each part: |error| <= 2^-24 a pass of the
state's norm, whatever the number of gates.

All lists, those held in FP32 among them, are no further off as gate programs than as tile
programs, which they are when a gate that mixes three qubits is in them (here XXX twice)."""
import math

import numpy as np
import pytest

from hiqsimulator_amd.circuits import H, Rx, Ry, Rz, X, haar_unitary, qft_like_circuit

pytestmark = pytest.mark.gpu

XXX = np.kron(np.kron(X, X), X)
CZ = np.diag([1, 1, 1, -1]).astype(np.complex128)


def layers(count, qubits, one, rng, two=None):
    out = []
    for layer in range(count):
        for q in qubits:
            out += [(m(float(rng.uniform(0, 2 * math.pi))), [q], []) for m in one]
        pairs = list(zip(qubits[layer % 2::2], qubits[layer % 2 + 1::2]))
        out += [(X, [b], [a]) if two is None else (two, [a, b], []) for a, b in pairs]
    return out


def ising(n, angles):
    out = []
    for zz, x in angles:
        out += [(np.diag(np.exp(1j * zz * np.array([1, -1, -1, 1]))), [i, i + 1], []) for i in range(n - 1)]
        out += [(Rx(x), [q], []) for q in range(n)]
    return out


def heisenberg(n, steps):
    out = []
    for _ in range(steps):
        for i in range(n - 1):
            hh = [(H, [i], []), (H, [i + 1], [])]
            out += hh + [(X, [i + 1], [i]), (Rz(0.3), [i + 1], []), (X, [i + 1], [i])] + hh
    return out


HELD_IN_FP64 = {
    "equal": lambda n, rng: layers(20, list(range(n)), [lambda _: Rx(0.7)], rng),
    "cz": lambda n, rng: layers(20, list(range(n)), [Ry], rng, CZ),
    "h and cz": lambda n, rng: layers(10, list(range(n)), [lambda _: H], rng, CZ),
    "haar": lambda n, rng: [(haar_unitary(2, rng), [q], []) for q in range(n)],
    "haar and cnot": lambda n, rng: layers(8, list(range(n)), [lambda _: haar_unitary(2, rng)], rng),
    "zyz": lambda n, rng: layers(10, list(range(n)), [Rz, Ry, Rz], rng),
    "zxzxz": lambda n, rng: layers(6, list(range(n)), [Rz, Rx, Rz, Rx, Rz], rng),
    "few": lambda n, rng: layers(200, [1, 5, n - 2, n // 2], [Ry, Rz], rng),
    "ising": lambda n, rng: ising(n, [(0.3, 0.4)] * 40),
    "qaoa": lambda n, rng: ising(n, rng.uniform(0.1, 1.5, (8, 2))),
    "heisenberg": lambda n, rng: heisenberg(n, 4),
}
HELD_IN_FP32 = {
    "rx": lambda n, rng: layers(20, list(range(n)), [Rx], rng),
    "small angles": lambda n, rng: layers(20, list(range(n)), [lambda t: Ry(0.01 * t)], rng),
    "controlled": lambda n, rng: [(Ry(0.3 + i), [int(q[0])], [int(q[1]), int(q[2])])
                                  for i in range(100) for q in [rng.permutation(n)[:3]]],
    "diagonal": lambda n, rng: [(np.diag(np.exp(1j * rng.uniform(0, 6, 8))), [int(p) for p in rng.permutation(n)[:3]], [])
                                for _ in range(60)],
    "qft": lambda n, rng: qft_like_circuit(n),
    "cnot": lambda n, rng: [(X, [i + 1], [i]) for _ in range(8) for i in range(n - 1)],
}


class Pair:
    """The same state in complex64 and complex128."""

    def __init__(self, engine_mod, n, zeros=False):
        ids = list(range(n))
        self.sims = [engine_mod.SimulatorMPI(1, n, 4, p) for p in ("c64", "c128")]
        for sim in self.sims:
            sim.allocate_qureg(ids, 0)
        if not zeros:
            self.sims[0].init_random_state(3)
            self.sims[1].set_wavefunction(self.sims[0].get_state(), ids)
        for sim in self.sims:
            sim.snapshot()

    def error(self, gates):
        for sim in self.sims:
            sim.restore()
        norm = np.linalg.norm(self.sims[1].get_state())
        passes = self.sims[0].apply_tiled(gates, 4)
        self.sims[1].apply_tiled(gates, 4)
        a, b = (sim.get_state() for sim in self.sims)
        return np.linalg.norm(a - b) / norm, passes


@pytest.mark.parametrize("n", [21, 22])
def test_rounding_does_not_grow_with_the_gates(engine_mod, n):
    pair = Pair(engine_mod, n)
    for name, make in HELD_IN_FP64.items():
        gates = make(n, np.random.default_rng(n))
        print("gate precision n=%d %s" % (n, name), flush=True)
        err, passes = pair.error(gates)
        # (1e-15 a gate for the complex128 side)
        assert err <= passes * 2.0 ** -24 + 1e-15 * len(gates), name


@pytest.mark.parametrize("zeros", [False, True])
def test_no_further_off_than_fused_products(engine_mod, zeros):
    """From |0..0> for the lists held in FP64: there most products are exact or nearly so."""
    n = 21
    pair = Pair(engine_mod, n, zeros)
    for name, make in (HELD_IN_FP64 if zeros else {**HELD_IN_FP64, **HELD_IN_FP32}).items():
        gates = make(n, np.random.default_rng(n))
        print("gates against products from zeros %d: %s" % (zeros, name), flush=True)
        err, _ = pair.error(gates)
        products, _ = pair.error(gates + [(XXX, [0, 1, 2], [])] * 2)
        # (both within 1e-9 where the products happen to be exact)
        assert err <= products + 1e-9, name
