"""Dense passes on small states (one thread per output amplitude) against
numpy, around the size where the other forms take over (2^18 amplitudes, 2^19
at k = 4), with targets in any order and controls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [5, 7, 9, 13, 18, 19, 20])
@pytest.mark.parametrize("k", [2, 3, 4, 5])
def test_small_dense(engine_mod, n, k, precision):
    rng = np.random.default_rng(100 * n + k)
    sim = engine_mod.SimulatorMPI(1, n, 5, precision)
    sim.allocate_qureg(list(range(n)), 0)
    sim.init_random_state(3)
    psi = np.asarray(sim.get_state())
    print("small dense n=%d k=%d %s" % (n, k, precision), flush=True)
    for controls in (0, 1, 2):
        if k + controls > n:
            continue
        perm = [int(p) for p in rng.permutation(n)]
        pos, ctrl = perm[:k], perm[k:k + controls]
        u, _ = np.linalg.qr(rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k)))
        sim.apply_matrix(u, pos, sum(1 << c for c in ctrl))
        v = psi.reshape((2,) * n)
        axes = [n - 1 - p for p in pos[::-1]]
        new = np.moveaxis(np.tensordot(u.reshape((2,) * (2 * k)), v, axes=(range(k, 2 * k), axes)), range(k), axes)
        i = np.arange(1 << n)
        on = np.all([(i >> c) & 1 == 1 for c in ctrl], axis=0) if ctrl else np.ones(1 << n, bool)
        psi = np.where(on, new.reshape(-1), psi)
    # 2 * 2^k roundings per output and pass, of amplitudes below 1
    assert np.abs(np.asarray(sim.get_state()) - psi).max() <= 3 * 2 ** (k + 2) * (2.0 ** -24 if precision == "c64" else 2.0 ** -53)
