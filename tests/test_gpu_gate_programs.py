"""Gate programs on the GPU against the oracle, at the sizes around a tile (2^13
amplitudes in complex128, 2^14 in complex64) and with every kind of record:
rotations, Hadamards, general one-qubit gates, phases and diagonals, swaps and
two-qubit unitaries, each plain and under controls, on bits of every place
(register, lane, wave, other tiles)."""
import math

import numpy as np
import pytest

from hiqsimulator_amd.batching import fidelity
from hiqsimulator_amd.circuits import H, R, Rx, Ry, Rz, S, X, Y, Z, apply_circuit_inorder, haar_unitary

pytestmark = pytest.mark.gpu

SWAP = np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], dtype=np.complex128)


def gates_of(n, count, seed, wide=False):
    rng = np.random.default_rng(seed)
    out = [(H, [q], []) for q in range(n)]
    for i in range(count):
        t = float(rng.uniform(0, 2 * math.pi))
        m = [H, Rx(t), Ry(t), Rz(t), R(t), X, Y, Z, S, haar_unitary(2, rng), SWAP, haar_unitary(4, rng),
             np.diag(np.exp(1j * rng.uniform(0, 6, 8))), np.kron(haar_unitary(2, rng), np.diag([1, 1j])),
             Ry(math.pi), Rx(math.pi)][i % 16]
        k = int(math.log2(len(m)))
        nc = int(rng.integers(0, 3)) if i % 3 == 0 else 0
        q = [int(p) for p in rng.permutation(n)[:k + nc]]
        out.append((m, q[:k], q[k:]))
    if wide:
        out.insert(len(out) // 2, (haar_unitary(8, rng), [n - 1, 0, 5], []))
    return out


def oracle_state(oracle_mod, n, gates):
    o = oracle_mod.OracleSim(1, n, 5)
    o.allocate_qureg(list(range(n)), 0)
    apply_circuit_inorder(o, gates, 5)
    return o.get_state()


@pytest.mark.parametrize("n", [12, 13, 14, 15, 17, 20, 21])
@pytest.mark.parametrize("flow", ["tiled", "run"])
def test_gate_programs_match_oracle(engine_mod, oracle_mod, n, flow):
    gates = gates_of(n, 64, 40 + n)
    ref = oracle_state(oracle_mod, n, gates)
    for prec in ("c128", "c64"):
        print("gate programs n=%d %s %s" % (n, flow, prec), flush=True)
        sim = engine_mod.SimulatorMPI(1, n, 5, prec)
        sim.allocate_qureg(list(range(n)), 0)
        if flow == "tiled":
            sim.apply_tiled(gates, 4)
        else:
            apply_circuit_inorder(sim, gates, 5)
        psi = sim.get_state()
        if prec == "c128":
            assert np.abs(psi - ref).max() <= 1e-12
        else:
            # 8 eps of the largest amplitude a gate, as in the host test
            assert np.abs(psi - ref).max() <= 8 * 2.0 ** -23 * len(gates) * np.abs(ref).max()
            assert fidelity(psi, ref) >= 1 - 1e-6


def test_three_mixed_qubits_take_tile_programs(engine_mod, oracle_mod):
    n = 15
    gates = gates_of(n, 40, 9, wide=True)
    print("tile programs n=%d" % n, flush=True)
    ref = oracle_state(oracle_mod, n, gates)
    for prec, tol in (("c128", 1e-12), ("c64", 8 * 2.0 ** -23 * len(gates) * np.abs(ref).max())):
        sim = engine_mod.SimulatorMPI(1, n, 5, prec)
        sim.allocate_qureg(list(range(n)), 0)
        sim.apply_tiled(gates, 4)
        assert np.abs(sim.get_state() - ref).max() <= tol


def test_long_gate_list_on_few_qubits(engine_mod, oracle_mod):
    """More stages than one pass holds, and phases of one qubit with every other one."""
    n = 13
    gates = [(H, [q], []) for q in range(n)]
    for i in range(700):
        gates.append((Ry(0.01 * i), [i % n], [(i + n - 1) % n]))
        if i % 70 == 0:
            gates += [(R(0.3 + m), [i % n], [m]) for m in range(n) if m != i % n]
    print("long list n=%d, %d gates" % (n, len(gates)), flush=True)
    sim = engine_mod.SimulatorMPI(1, n, 5)
    sim.allocate_qureg(list(range(n)), 0)
    assert sim.apply_tiled(gates, 4) >= 1
    assert np.abs(sim.get_state() - oracle_state(oracle_mod, n, gates)).max() <= 1e-12


@pytest.mark.parametrize("n", [13, 14, 15, 18, 21])
@pytest.mark.parametrize("pinned", [False, True])
def test_last_pass_permutes(engine_mod, oracle_mod, n, pinned):
    """Permutations right behind queued gates: the last pass stores the state
    permuted where its tile has room, and a pass of its own does where not."""
    rng = np.random.default_rng(n)
    parts = [gates_of(n, c, 60 + n + c) for c in (3, 16, 40)]
    perms = [[int(q) for q in rng.permutation(n)] for _ in range(3)]
    perms[1] = perms[1][:4] + sorted(perms[1][4:])
    ref = oracle_state(oracle_mod, n, [g for part in parts for g in part])
    # ids are qubits: the state's bit p holds qubit perms[-1][p]
    i, src = np.arange(1 << n), np.zeros(1 << n, dtype=np.int64)
    for p, q in enumerate(perms[-1]):
        src |= ((i >> p) & 1) << q
    ref = ref[src]
    for prec in ("c128", "c64"):
        print("permuting passes n=%d %s pinned=%d" % (n, prec, pinned), flush=True)
        sim = engine_mod.SimulatorMPI(1, n, 5, prec)
        sim.allocate_qureg(list(range(n)), 0)
        view = sim.state_dlpack() if pinned else None  # results go back into the viewed buffer
        for gates, order in zip(parts, perms):
            apply_circuit_inorder(sim, gates, 5)
            sim.permute_qubits(order)
        sim.synchronize()
        psi = sim.get_state()
        tol = 1e-12 if prec == "c128" else 8 * 2.0 ** -23 * sum(map(len, parts)) * np.abs(ref).max()
        assert np.abs(psi - ref).max() <= tol
        del view
