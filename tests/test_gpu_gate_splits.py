"""Gate programs on states of 1 GiB and more, where the stages of a pass are split in the best of
four ways, against the same list as tile programs (which it is when a gate that mixes three
qubits is in it, here XXX twice)."""
import math

import numpy as np
import pytest

from hiqsimulator_amd.circuits import H, R, Rx, Ry, X, haar_unitary

pytestmark = pytest.mark.gpu

XXX = np.kron(np.kron(X, X), X)


def gates_of(n, seed):
    """Every kind of record on bits of every place, then layers that fill whole passes; with seed 1 and
    27 qubits the four ways save two stages of 36 in complex128 and three of 29 in complex64."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(48):
        t = float(rng.uniform(0, 2 * math.pi))
        m = [H, Rx(t), Ry(t), R(t), haar_unitary(2, rng), haar_unitary(4, rng), np.diag(np.exp(1j * rng.uniform(0, 6, 8))),
             np.kron(haar_unitary(2, rng), np.diag([1, 1j]))][i % 8]
        k = int(math.log2(len(m)))
        q = [int(p) for p in rng.permutation(n)[:k + i % 3]]
        out.append((m, q[:k], q[k:]))
    for layer in range(8):
        out += [(Ry(float(t)), [q], []) for q, t in enumerate(rng.uniform(0, 6, n))]
        out += [(X, [q + 1], [q]) for q in range(layer % 2, n - 1, 2)]
    return out


@pytest.mark.parametrize("n,prec", [(27, "c128"), (27, "c64")])
def test_split_passes_match_tile_programs(engine_mod, n, prec):
    gates = gates_of(n, 1)
    print("split passes n=%d %s" % (n, prec), flush=True)
    sim = engine_mod.SimulatorMPI(1, n, 4, prec)
    sim.allocate_qureg(list(range(n)), 0)
    sim.init_random_state(7)
    sim.snapshot()
    norm = np.linalg.norm(sim.get_state())
    sim.apply_tiled(gates, 4)
    psi = sim.get_state()
    sim.restore()
    sim.apply_tiled(gates + [(XXX, [0, 1, 2], [])] * 2, 4)
    psi -= sim.get_state()
    # 8 eps of the state's norm a gate, as for smaller states
    eps = 2.0 ** -52 if prec == "c128" else 2.0 ** -23
    assert np.linalg.norm(psi) <= 8 * eps * len(gates) * norm
