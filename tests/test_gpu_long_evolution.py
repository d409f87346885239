"""Long time evolutions from a state at the spectrum's edge (the ground state of a
commuting sum with positive terms), where exp(-i t H) is a phase: the Chebyshev
recurrence must neither grow there nor lose more than the Taylor steps would.

Bound: a unit of reach |t| sum|c| in Taylor steps takes a rounding of the weights and
fifteen sums, each up to eps of the amplitude: 16 eps a unit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# sums whose reciprocal rounds up in FP32: 2 / sum times the sum is above 2
SCALES = [0.37, 0.61, 0.83, 0.97]


def coefficients(count, scale):
    c = np.linspace(0.4, 1.0, count) * scale
    while float(np.float32(2 / c.sum())) * float(np.float32(c.sum())) <= 2 * (1 + 2.0 ** -25):
        c = c * 1.0137
    return [float(x) for x in c]


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("kind", ["zz", "x", "controlled"])
def test_phase_of_an_edge_state(engine_mod, kind, scale):
    n = 10
    ids = list(range(n))
    for precision, eps in (("c64", 2.0 ** -24), ("c128", 2.0 ** -53)):
        for reach in (40.0, 255.9, 257.0, 5e4):
            print("long evolution %s %s reach %g" % (kind, precision, reach), flush=True)
            sim = engine_mod.SimulatorMPI(1, n, 4, precision)
            sim.allocate_qureg(ids, 0)
            ctrls = []
            if kind == "x":
                c = coefficients(n, scale)
                terms = [([(q, "X")], c[q]) for q in ids]
                ref = np.full(1 << n, 2.0 ** (-n / 2), dtype=np.complex128)
            else:
                m = n - 1 if kind == "controlled" else n  # the last qubit is the control
                c = coefficients(m - 1, scale)
                terms = [([(q, "Z"), (q + 1, "Z")], c[q]) for q in range(m - 1)]
                ref = np.zeros(1 << n, dtype=np.complex128)
                ref[0] = 1
                if kind == "controlled":
                    ctrls = [n - 1]
                    ref[0] = ref[1 << (n - 1)] = 0.5 ** 0.5
            sim.set_wavefunction(ref, ids)
            t = reach / sum(c)
            sim.emulate_time_evolution(terms, t, [q for q in ids if q not in ctrls], ctrls)
            phase = np.exp(-1j * t * sum(c))
            if kind == "controlled":
                ref[1 << (n - 1)] *= phase
            else:
                ref *= phase
            # + the rounding of the state given, and of the phase at 5e4 in FP64
            tol = np.linalg.norm(ref) * (16 * eps * (reach + 1) + 2.0 ** -52 * reach)
            assert np.linalg.norm(sim.get_state() - ref) <= tol, (precision, reach)
