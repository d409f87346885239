"""Long complex64 gate lists against the same lists in complex128: many gates a qubit, the same
angles again and again, long runs on few qubits.  On 21 and 22 qubits they run as gate programs,
which round each amplitude once a pass, by 2^-24 of each part: |error| <= 2^-24 a pass of the
state's norm, whatever the number of gates."""
import math

import numpy as np
import pytest

from hiqsimulator_amd.circuits import H, Rx, Ry, Rz, X

pytestmark = pytest.mark.gpu


def layers(n, count, qubits, one, rng):
    out = []
    for layer in range(count):
        for q in qubits:
            out += [(m(float(rng.uniform(0, 2 * math.pi))), [q], []) for m in one]
        out += [(X, [b], [a]) for a, b in zip(qubits[layer % 2::2], qubits[layer % 2 + 1::2])]
    return out


def ising(n, steps):
    zz = np.diag(np.exp(0.3j * np.array([1, -1, -1, 1])))
    return [g for _ in range(steps) for g in [(zz, [i, i + 1], []) for i in range(n - 1)] +
            [(Rx(0.4), [q], []) for q in range(n)]]


def heisenberg(n, steps):
    out = []
    for _ in range(steps):
        for i in range(n - 1):
            hh = [(H, [i], []), (H, [i + 1], [])]
            out += hh + [(X, [i + 1], [i]), (Rz(0.3), [i + 1], []), (X, [i + 1], [i])] + hh
    return out


@pytest.mark.parametrize("n", [21, 22])
@pytest.mark.parametrize("kind", ["layers", "zyz", "zxzxz", "few", "ising", "heisenberg"])
def test_rounding_does_not_grow_with_the_gates(engine_mod, n, kind):
    rng = np.random.default_rng(n)
    qubits = list(range(n))
    gates = {"layers": lambda: layers(n, 30, qubits, [Rx], rng),
             "zyz": lambda: layers(n, 10, qubits, [Rz, Ry, Rz], rng),
             "zxzxz": lambda: layers(n, 6, qubits, [Rz, Rx, Rz, Rx, Rz], rng),
             "few": lambda: layers(n, 200, [1, 5, n - 2, n // 2], [Ry, Rz], rng),
             "ising": lambda: ising(n, 40),
             "heisenberg": lambda: heisenberg(n, 4)}[kind]()
    sims = []
    for precision in ("c64", "c128"):
        sim = engine_mod.SimulatorMPI(1, n, 4, precision)
        sim.allocate_qureg(qubits, 0)
        sims.append(sim)
    sims[0].init_random_state(3)
    start = sims[0].get_state()
    sims[1].set_wavefunction(start, qubits)
    passes = [sim.apply_tiled(gates, 4) for sim in sims]
    print("gate precision n=%d %s: %d gates, %s passes" % (n, kind, len(gates), passes), flush=True)
    got, ref = (sim.get_state() for sim in sims)
    # (1e-15 a gate for the complex128 side)
    assert np.linalg.norm(got - ref) <= np.linalg.norm(start) * (passes[0] * 2.0 ** -24 + 1e-15 * len(gates))
