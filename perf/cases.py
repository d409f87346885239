"""The work that users of the simulator have it do, as cases that can be timed.

A case is a dict of plain values; ``kind`` says which user's call it is:

  session   one ProjectQ-style program on a kept simulator: allocate, gates cluster by
            cluster (what the GreedyScheduler sends), one amplitude, one probability, the
            whole state (cheat), measure every qubit, deallocate every qubit.  Small
            states: latency, launches and host work count.
  circuit   a long random circuit on a resident state, cluster by cluster through
            apply_controlled_gate and run(), with qubit permutations in between (the
            benchmark's flow; `flow` "run"), or as one gate list through apply_tiled
            (`flow` "tiled").
  qft       the quantum Fourier transform (H and controlled phases), run() per cluster.
  passes    one fused pass per run() (pass mode 0, the reference's own way): dense
            unitaries on 1 to 5 qubits, a diagonal one, gates under a control mask.
  expect    the expectation value of a Hamiltonian (a Pauli sum), as in VQE.
  evolve    emulate_time_evolution under a Hamiltonian, then apply_qubit_operator, from
            the state's snapshot.
  readout   probabilities, entropy, a collapse, a measurement and a permutation of a
            large state taken back from its snapshot.
  sample    computational-basis shots of a large state.
  batch     many uneven circuits in one graph launch, every final state fetched.
  serve     a burst of requests (samples or expectation values) through the request loop.

Precisions are the engine's two, "c128" and "c64".  States that are given are normalised
complex Gaussian vectors, which is what deep random circuits leave behind.
"""
import math

import numpy as np
import torch

from hiqsimulator_amd import SimulatorMPI, state_view
from hiqsimulator_amd.batching import load_tuning, make_batch
from hiqsimulator_amd.scheduling import plan_clusters
from hiqsimulator_amd.serving import make_server

CLUSTER = 4  # fusion width of the benchmark's headline


def listed():
    return [
        # A toy program in a notebook or a test: every call is latency.
        {"name": "session-6q", "kind": "session", "n": 6, "layers": 8, "prec": "c128"},
        # The 16-qubit plain-method configuration: a 1 MiB state.
        {"name": "session-16q", "kind": "session", "n": 16, "layers": 20, "prec": "c128"},
        # The headline configuration: 30 qubits, 40 layers, 8 permutations, complex128.
        {"name": "circuit-30q", "kind": "circuit", "flow": "run", "n": 30, "layers": 40, "perms": 8, "prec": "c128"},
        # A medium state in single precision, the whole gate list at once.
        {"name": "circuit-23q-c64", "kind": "circuit", "flow": "tiled", "n": 23, "layers": 20, "perms": 0, "prec": "c64"},
        # The precision configuration's QFT, at a size whose reference fits beside it.
        {"name": "qft-29q-c64", "kind": "qft", "n": 29, "prec": "c64"},
        # The reference's own way: one HBM pass per run(), all widths, diagonal and controlled.
        {"name": "passes-27q", "kind": "passes", "n": 27, "count": 14, "prec": "c128"},
        # VQE energy: Heisenberg chain with a field, 101 terms.
        {"name": "expect-26q", "kind": "expect", "n": 26, "ham": "heisenberg", "terms": 0, "prec": "c128"},
        # Trotter-free dynamics: transverse-field Ising chain.
        {"name": "evolve-20q", "kind": "evolve", "n": 20, "ham": "ising", "terms": 0, "time": 0.25, "prec": "c128"},
        # Mid-circuit measurement and analysis of a large state.
        {"name": "readout-28q", "kind": "readout", "n": 28, "prec": "c128"},
        # Shots of a large state, the request size of the serving configuration.
        {"name": "sample-28q-c64", "kind": "sample", "n": 28, "shots": 1024, "prec": "c64"},
        # Uneven circuits as in the batching configuration, in the number whose states one fetches.
        {"name": "batch-48-c64", "kind": "batch", "count": 48, "lo": 10, "hi": 18, "depth": 40, "prec": "c64"},
        # A burst of the serving configuration's requests.
        {"name": "serve-24-c64", "kind": "serve", "count": 24, "lo": 12, "hi": 24, "depth": 40, "prec": "c64"},
    ]


def draw(rng):
    kind = rng.choice(["session", "circuit", "qft", "passes", "expect", "evolve", "readout", "sample", "batch", "serve"])
    prec = rng.choice(["c128", "c64"])
    if kind == "session":
        return {"kind": kind, "n": rng.randint(4, 18), "layers": rng.randint(4, 24), "prec": prec}
    if kind == "circuit":
        n = rng.randint(17, 29)
        return {"kind": kind, "flow": rng.choice(["run", "tiled"]), "n": n, "layers": rng.randint(8, 40),
                "perms": rng.choice([0, 0, 1, 3, 8]), "prec": prec}
    if kind == "qft":
        return {"kind": kind, "n": rng.randint(14, 29), "prec": prec}
    if kind == "passes":
        return {"kind": kind, "n": rng.randint(13, 28), "count": rng.randint(7, 21), "prec": prec}
    if kind == "expect":
        return {"kind": kind, "n": rng.randint(11, 27), "ham": rng.choice(["heisenberg", "ising", "random"]),
                "terms": rng.randint(1, 120), "prec": prec}
    if kind == "evolve":
        return {"kind": kind, "n": rng.randint(9, 21), "ham": rng.choice(["heisenberg", "ising", "random"]),
                "terms": rng.randint(2, 40), "time": round(rng.uniform(0.02, 0.3), 3), "prec": prec}
    if kind == "readout":
        return {"kind": kind, "n": rng.randint(16, 28), "prec": prec}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(15, 29), "shots": int(2 ** rng.uniform(3, 15)), "prec": prec}
    if kind == "batch":
        lo = rng.randint(6, 14)
        return {"kind": kind, "count": rng.randint(12, 60), "lo": lo, "hi": lo + rng.randint(0, 4),
                "depth": rng.randint(12, 60), "prec": prec}
    lo = rng.randint(10, 18)
    return {"kind": kind, "count": rng.randint(6, 30), "lo": lo, "hi": lo + rng.randint(1, 7),
            "depth": rng.randint(20, 60), "prec": prec}


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------
H = np.array([[1, 1], [1, -1]], dtype=np.complex128) / math.sqrt(2.0)
X = np.array([[0, 1], [1, 0]], dtype=np.complex128)


def rotation(kind, t):
    c, s = math.cos(t / 2), math.sin(t / 2)
    if kind == 0:
        return H
    if kind == 1:
        return np.array([[c, -1j * s], [-1j * s, c]])
    if kind == 2:
        return np.array([[c, -s], [s, c]], dtype=np.complex128)
    return np.array([[c - 1j * s, 0], [0, c + 1j * s]])


def haar(dim, rng):
    q, r = np.linalg.qr(rng.normal(size=(dim, dim)) + 1j * rng.normal(size=(dim, dim)))
    d = np.diag(r)
    return q * (d / np.abs(d))


def layered(n, layers, rng, haar_every=0):
    """H or a random rotation on every qubit, then CNOTs between neighbours; layer by layer."""
    out = []
    for layer in range(layers):
        gates = [(rotation(int(k), float(t)), [q], []) for q, (k, t) in
                 enumerate(zip(rng.integers(0, 4, size=n), rng.uniform(0, 2 * math.pi, size=n)))]
        gates += [(X, [i + 1], [i]) for i in range(layer % 2, n - 1, 2)]
        if haar_every and n > 1 and (layer + 1) % haar_every == 0:
            a, b = rng.choice(n, size=2, replace=False)
            gates.append((haar(4, rng), [int(a), int(b)], []))
        out.append(gates)
    return out


def flat(layers):
    return [g for layer in layers for g in layer]


def circuit_steps(case, rng):
    """[("gates", list) | ("perm", ids), ...]"""
    n, layers, perms = case["n"], case["layers"], case["perms"]
    made = layered(n, layers, rng)
    stride = max(1, layers // perms) if perms else layers + 1
    steps, cur, left = [], [], perms
    for i, gates in enumerate(made):
        cur += gates
        if left and (i + 1) % stride == 0:
            steps += [("gates", cur), ("perm", [int(q) for q in rng.permutation(n)])]
            cur, left = [], left - 1
    if cur:
        steps.append(("gates", cur))
    return steps


def qft_gates(n, seed):
    """The QFT on a register whose qubits come in the seed's rotated order."""
    order = [(q + seed) % n for q in range(n)]
    gates = []
    for j in reversed(range(n)):
        gates.append((H, [order[j]], []))
        for m in reversed(range(j)):
            p = np.array([[1, 0], [0, np.exp(2j * math.pi / 2 ** (j - m + 1))]])
            gates.append((p, [order[j]], [order[m]]))
    return gates


def pass_gates(case, rng):
    """Widths 1 to 5 in turn, then a diagonal gate and one under a control mask."""
    n, out = case["n"], []
    for i in range(case["count"]):
        q = [int(p) for p in rng.permutation(n)]
        if i % 7 < 5:
            k = i % 7 + 1
            out.append((haar(1 << k, rng), q[:k], []))
        elif i % 7 == 5:
            out.append((np.diag(np.exp(2j * math.pi * rng.random(8))), q[:3], []))
        else:
            out.append((haar(8, rng), q[:3], q[3:6]))  # 3 targets, 3 controls: wider than a cluster
    return out


def hamiltonian(case, rng):
    """[([(qubit, "X" | "Y" | "Z"), ...], coefficient), ...]"""
    n, kind = case["n"], case["ham"]
    c = lambda: float(rng.uniform(0.2, 1.0))  # noqa: E731
    if kind == "heisenberg":
        terms = [([(i, p), (i + 1, p)], c()) for i in range(n - 1) for p in "XYZ"]
        return terms + [([(i, "Z")], c()) for i in range(n)]
    if kind == "ising":
        return [([(i, "Z"), (i + 1, "Z")], c()) for i in range(n - 1)] + [([(i, "X")], c()) for i in range(n)]
    terms = []
    for _ in range(case["terms"]):
        qs = sorted(int(q) for q in rng.choice(n, size=int(rng.integers(1, min(4, n) + 1)), replace=False))
        terms.append(([(q, "XYZ"[int(rng.integers(3))]) for q in qs], c()))
    return terms


def qubit_operator(n, rng):
    """The short operator that is applied after an evolution (an observable's perturbation)."""
    a, b = (int(q) for q in rng.choice(n, size=2, replace=False))
    return [([], 0.6), ([(a, "X")], 0.5), ([(a, "Z"), (b, "Y")], 0.25)]


def small_circuits(case, rng):
    """Sizes spread over lo..hi and depths over depth/3..depth, in an uneven order; the gates are the seed's."""
    lo, hi, count, depth = case["lo"], case["hi"], case["count"], case["depth"]
    out = []
    for i in range(count):
        n = lo + (5 * i) % (hi - lo + 1)
        d = max(4, depth // 3) + (7 * i) % (depth - max(4, depth // 3) + 1)
        out.append((n, flat(layered(n, d, rng, haar_every=5))))
    return out


def requests(case, rng):
    """Sizes log-spread over lo..hi and depths over 20..depth, in an uneven order; samples and expectations in turn."""
    lo, hi, count = math.log(case["lo"]), math.log(case["hi"] + 1), case["count"]
    out = []
    for i in range(count):
        n = min(case["hi"], int(math.exp(lo + (hi - lo) * ((i * 0.6180339887) % 1.0))))
        gates = flat(layered(n, 20 + (7 * i) % (case["depth"] - 19), rng))
        if i % 2 == 0:
            out.append({"n": n, "gates": gates, "shots": 1024, "seed": int(rng.integers(1 << 62))})
        else:
            terms = []
            for _ in range(8):
                x = z = 0
                for q in rng.choice(n, size=int(rng.integers(1, 5)), replace=False):
                    p = int(rng.integers(3))
                    x |= (p < 2) << int(q)
                    z |= (p > 0) << int(q)
                terms.append((x, z))
            out.append({"n": n, "gates": gates, "terms": terms})
    return out


def fill_random(psi, seed):
    """A normalised complex Gaussian state into the tensor psi."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    chunk = 1 << 26
    norm = 0.0
    for part in psi.split(chunk):
        part.copy_(torch.randn(part.numel(), dtype=torch.complex128, device="cuda", generator=g))
        norm = norm + torch.view_as_real(part).double().square().sum()
    for part in psi.split(chunk):
        part.mul_((1.0 / norm.sqrt()).to(part.dtype))


def simulator(case, seed, cluster=CLUSTER):
    n = case["n"]
    sim = SimulatorMPI(seed, n, cluster, case["prec"])
    sim.allocate_qureg(list(range(n)), 0)
    fill_random(state_view(sim), seed)
    torch.cuda.synchronize()
    return sim


def planned(gates, n, k=CLUSTER):
    return [[gates[i] for i in c] for c in plan_clusters(gates, list(range(n)), k, mode="lookahead")]


# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, n = case["kind"], case.get("n")
    rng = np.random.default_rng(seed)
    if kind == "session":
        gates = flat(layered(n, case["layers"], rng))
        bits = [bool(b) for b in rng.integers(0, 2, size=n)]
        return {"kind": kind, "n": n, "sim": SimulatorMPI(seed, n, CLUSTER, case["prec"]),
                "clusters": planned(gates, n), "bits": bits}
    if kind == "circuit":
        steps = circuit_steps(case, rng)
        if case["flow"] == "run":
            steps = [(k, planned(p, n) if k == "gates" else p) for k, p in steps]
        return {"kind": kind, "flow": case["flow"], "sim": simulator(case, seed), "steps": steps}
    if kind == "qft":
        return {"kind": kind, "sim": simulator(case, seed), "clusters": planned(qft_gates(n, seed), n)}
    if kind == "passes":
        sim = simulator(case, seed, cluster=5)
        sim.set_pass_mode(0)
        return {"kind": kind, "sim": sim, "gates": pass_gates(case, rng)}
    if kind == "expect":
        return {"kind": kind, "n": n, "sim": simulator(case, seed), "terms": hamiltonian(case, rng)}
    if kind == "evolve":
        sim = simulator(case, seed)
        sim.snapshot()
        return {"kind": kind, "n": n, "sim": sim, "terms": hamiltonian(case, rng), "time": case["time"],
                "op": qubit_operator(n, rng)}
    if kind == "readout":
        sim = simulator(case, seed)
        sim.snapshot()
        return {"kind": kind, "n": n, "sim": sim, **readout_plan(n, rng)}
    if kind == "sample":
        return {"kind": kind, "sim": simulator(case, seed), "shots": case["shots"], "seed": seed}
    if kind == "batch":
        t = load_tuning(case["prec"])
        b = make_batch(small_circuits(case, rng), case["prec"], t["k_by_n"], t["wg_max_qubits"],
                       tile_min_qubits=t["tile_min_qubits"], prog_min_qubits=t["prog_min_qubits"])
        return {"kind": kind, "batch": b}
    server = make_server(case["prec"], state_bytes=12 << 30, matrix_bytes=1 << 30)
    return {"kind": kind, "server": server, "requests": requests(case, rng)}


def readout_plan(n, rng):
    q = [int(p) for p in rng.permutation(n)]
    return {"ask": q[:3], "values": [bool(b) for b in rng.integers(0, 2, size=3)], "collapse": q[3:4],
            "measure": q[4:6], "order": [int(p) for p in rng.permutation(n)]}


def run(state):
    kind = state["kind"]
    sim = state.get("sim")
    if kind == "session":
        n = state["n"]
        ids = list(range(n))
        sim.allocate_qureg(ids, 0)
        run_clusters(sim, state["clusters"])
        amp = sim.get_amplitude(state["bits"], ids)
        prob = sim.get_probability(state["bits"][:2], ids[:2])
        psi = sim.get_state()
        bits = sim.measure_qubits(ids)
        for q in ids:
            sim.deallocate_qubit(q)
        return {"amplitude": np.array([amp]), "probability": prob, "state": psi, "bits": np.array(bits)}
    if kind == "circuit":
        for what, payload in state["steps"]:
            if what == "perm":
                sim.permute_qubits(payload)
            elif state["flow"] == "run":
                run_clusters(sim, payload)
            else:
                sim.apply_tiled(payload, CLUSTER)
        return state_view(sim)
    if kind == "qft":
        run_clusters(sim, state["clusters"])
        return state_view(sim)
    if kind == "passes":
        for m, t, c in state["gates"]:
            sim.apply_controlled_gate(m, t, c)
            sim.run()
        return state_view(sim)
    if kind == "expect":
        return sim.get_expectation_value(state["terms"], list(range(state["n"])))
    if kind == "evolve":
        sim.restore()  # the operator does not keep the norm
        ids = list(range(state["n"]))
        sim.emulate_time_evolution(state["terms"], state["time"], ids, [])
        sim.apply_qubit_operator(state["op"], ids)
        return state_view(sim)
    if kind == "readout":
        sim.restore()
        prob = sim.get_probability(state["values"], state["ask"])
        entropy = sim.entropy()
        sim.collapse_wavefunction(state["collapse"], state["values"][:1])
        bits = sim.measure_qubits(state["measure"])
        sim.permute_qubits(state["order"])
        return {"probability": prob, "entropy": entropy, "bits": np.array(bits), "state": state_view(sim)}
    if kind == "sample":
        return sim.sample(state["shots"], state["seed"]).view(np.int64)
    if kind == "batch":
        b = state["batch"]
        b.run()
        return [b.get_state(i) for i in range(len(b))]
    server = state["server"]
    ids = []
    for r in state["requests"]:
        if "shots" in r:
            ids.append(server.submit_samples(r["n"], r["gates"], r["shots"], r["seed"]))
        else:
            ids.append(server.submit_expectation(r["n"], r["gates"], [x for x, _ in r["terms"]], [z for _, z in r["terms"]]))
    left = len(ids)
    while left:
        left -= len(server.step(block=True))
    out = []
    for i, r in zip(ids, state["requests"]):
        out.append(server.samples(i).view(np.int64) if "shots" in r else server.expectations(i))
        server.forget(i)
    return out


def run_clusters(sim, clusters):
    for cluster in clusters:
        for m, t, c in cluster:
            sim.apply_controlled_gate(m, t, c)
        sim.run()


# ---------------------------------------------------------------------------
def gate_flops(m, t, c, n):
    """Real operations of one gate applied by itself: none for a permutation, one complex
    product an amplitude for a diagonal, the dense product otherwise."""
    if np.count_nonzero(m) == len(m):
        return 0 if np.all(np.isin(m, (0, 1))) else 6 << (n - len(c))
    return 8 << (len(t) + n - len(c))


def work(case):
    kind, n = case["kind"], case.get("n")
    amp = 16 if case["prec"] == "c128" else 8
    rng = np.random.default_rng(1)
    size = amp << n if n else 0
    count = lambda gates, q: float(sum(gate_flops(m, t, c, q) for m, t, c in gates))  # noqa: E731
    if kind == "session":  # the state comes to the host in complex128
        return {"bytes": float(16 << n), "flops": count(flat(layered(n, case["layers"], rng)), n)}
    if kind == "circuit":
        return {"bytes": 2.0 * size, "flops": count(flat(layered(n, case["layers"], rng)), n)}
    if kind == "qft":
        return {"bytes": 2.0 * size, "flops": count(qft_gates(n, 1), n)}
    if kind == "passes":
        gates = pass_gates(case, rng)
        return {"bytes": 2.0 * size * sum(2.0 ** -len(c) for _, _, c in gates), "flops": count(gates, n)}
    if kind == "expect":
        return {"bytes": float(size), "flops": 8.0 * len(hamiltonian(case, rng)) * 2 ** n}
    if kind == "evolve":
        terms = hamiltonian(case, rng)
        return {"bytes": 2.0 * size, "flops": 8.0 * taylor_products(terms, case["time"]) * len(terms) * 2 ** n}
    if kind == "readout":
        return {"bytes": 2.0 * size, "flops": 10.0 * 2 ** n}
    if kind == "sample":
        return {"bytes": float(size + 8 * case["shots"]), "flops": 4.0 * 2 ** n}
    if kind == "batch":
        circuits = small_circuits(case, rng)
        return {"bytes": float(sum(16 << q for q, _ in circuits)), "flops": sum(count(g, q) for q, g in circuits)}
    reqs = requests(case, rng)
    return {"bytes": float(sum(amp << r["n"] for r in reqs)), "flops": sum(count(r["gates"], r["n"]) for r in reqs)}


def taylor_products(terms, time, tol=1e-12):
    """Products with the Hamiltonian that a Taylor series of exp(-i t H) takes to `tol`, in steps of unit norm."""
    norm = abs(time) * sum(abs(c) for _, c in terms)
    steps = max(1, math.ceil(norm))
    x, k, term = norm / steps, 0, 1.0
    while term > tol and k < 64:
        k += 1
        term *= x / k
    return steps * k


# ---------------------------------------------------------------------------
# The same in plain torch, complex128
# ---------------------------------------------------------------------------
def axes(psi, n, bits):
    """psi as a view with one axis of length 2 per bit of `bits`, those axes in front, in the order given."""
    shape, at, top = [], {}, n
    for b in sorted(bits, reverse=True):
        shape += [1 << (top - b - 1), 2]
        at[b] = len(shape) - 1
        top = b
    shape.append(1 << top)
    return psi.view(shape).movedim([at[b] for b in bits], list(range(len(bits))))


def apply_gate(psi, n, m, targets, controls):
    v = axes(psi, n, list(controls) + list(reversed(targets)))
    for _ in controls:
        v = v[1]
    k = len(targets)
    if k == 1:
        a, b = v[0], v[1]
        t = a.clone()
        if m[0, 1] == 0 and m[1, 0] == 0:
            a.mul_(complex(m[0, 0]))
            b.mul_(complex(m[1, 1]))
            return
        a.mul_(complex(m[0, 0])).add_(b, alpha=complex(m[0, 1]))
        b.mul_(complex(m[1, 1])).add_(t, alpha=complex(m[1, 0]))
        return
    x = v.reshape(1 << k, -1)
    y = torch.as_tensor(np.ascontiguousarray(m), device=psi.device) @ x
    v.copy_(y.view(v.shape))


def parity_sign(i, z):
    """(-1)^popcount(i & z) as float64."""
    p = i & z
    for s in (32, 16, 8, 4, 2, 1):
        p = p ^ (p >> s)
    return 1.0 - 2.0 * (p & 1).double()


def apply_pauli(psi, idx, x, z):
    """P psi with P the product of i^{x & z} X^x Z^z over the qubits."""
    src = idx ^ x if x else idx
    v = psi[src] if x else psi.clone()
    if z:
        v *= parity_sign(src, z)
    return v * (1j ** (bin(x & z).count("1") % 4))


def masks(term):
    x = z = 0
    for q, p in term:
        x |= (p in "XY") << q
        z |= (p in "YZ") << q
    return x, z


def start_state(case, seed):
    psi = torch.empty(1 << case["n"], dtype=torch.complex128 if case["prec"] == "c128" else torch.complex64, device="cuda")
    fill_random(psi, seed)
    return psi.to(torch.complex128)


def zero_state(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1
    return psi


def permuted(psi, n, order, new):
    """The state whose bit p is the qubit new[p], from one whose bit p is order[p]."""
    at = {q: p for p, q in enumerate(order)}
    j = torch.arange(1 << n, device=psi.device)
    i = torch.zeros_like(j)
    for p, q in enumerate(new):
        i |= (j >> p & 1) << at[q]
    return psi[i]


def first_draw(seed):
    """The first uniform double of std::uniform_real_distribution over std::mt19937(seed)."""
    lo, hi = (int(v) for v in np.random.RandomState(seed).randint(0, 1 << 32, size=2, dtype=np.uint32))
    return (lo + hi * 4294967296.0) / 18446744073709551616.0


def pick(psi, u):
    """The first index whose running probability reaches u."""
    p = psi.real.square() + psi.imag.square()
    rows = p.view(-1, min(p.numel(), 1 << 12))
    ends = torch.cumsum(rows.sum(1), 0)
    r = int(torch.searchsorted(ends, torch.tensor(u, dtype=torch.float64, device=psi.device)))
    r = min(r, rows.shape[0] - 1)
    before = float(ends[r - 1]) if r else 0.0
    c = int(torch.searchsorted(torch.cumsum(rows[r], 0) + before, torch.tensor(u, dtype=torch.float64, device=psi.device)))
    return r * rows.shape[1] + min(c, rows.shape[1] - 1)


def exact(case, seed):
    kind, n = case["kind"], case.get("n")
    rng = np.random.default_rng(seed)
    if kind == "session":
        psi = zero_state(n)
        for m, t, c in flat(layered(n, case["layers"], rng)):
            apply_gate(psi, n, m, t, c)
        bits = rng.integers(0, 2, size=n)
        at = sum(int(b) << q for q, b in enumerate(bits))
        p = axes(psi, n, [0, 1])[int(bits[0]), int(bits[1])]
        return {"amplitude": psi[at].reshape(1), "probability": float(torch.view_as_real(p.contiguous()).square().sum()),
                "state": psi, "bits": None}
    if kind == "circuit":
        if case["layers"] * n * 2.0 ** n > 40 * 28 * 2.0 ** 28:
            return None  # over 20 seconds
        psi, order = start_state(case, seed), list(range(n))
        for what, payload in circuit_steps(case, rng):
            if what == "perm":
                psi = permuted(psi, n, order, payload)
                order = payload
                continue
            at = {q: p for p, q in enumerate(order)}
            for m, t, c in payload:
                apply_gate(psi, n, m, [at[q] for q in t], [at[q] for q in c])
        return psi
    if kind == "qft":
        psi = start_state(case, seed)
        for m, t, c in qft_gates(n, seed):
            apply_gate(psi, n, m, t, c)
        return psi
    if kind == "passes":
        psi = start_state(case, seed)
        for m, t, c in pass_gates(case, rng):
            apply_gate(psi, n, m, t, c)
        return psi
    if kind in ("expect", "evolve"):
        psi = start_state(case, seed)
        idx = torch.arange(1 << n, device="cuda")
        terms = [masks(t) + (c,) for t, c in hamiltonian(case, rng)]
        if kind == "expect":
            return sum(c * float(torch.view_as_real(psi).mul(torch.view_as_real(apply_pauli(psi, idx, x, z))).sum()) for x, z, c in terms)
        norm = abs(case["time"]) * sum(abs(c) for _, _, c in terms)
        steps = max(1, math.ceil(norm))
        for _ in range(steps):
            a, out = psi, psi.clone()
            for k in range(1, 40):
                b = torch.zeros_like(a)
                for x, z, c in terms:
                    b += apply_pauli(a, idx, x, z) * (-1j * case["time"] / steps * c / k)
                out += b
                a = b
                if float(a.abs().square().sum()) < 1e-32:
                    break
            psi = out
        return sum(apply_pauli(psi, idx, x, z) * c for x, z, c in (masks(t) + (c,) for t, c in qubit_operator(n, rng)))
    if kind == "readout":
        psi, plan = start_state(case, seed), readout_plan(n, rng)
        p = psi.real.square() + psi.imag.square()
        prob = float(axes(p, n, plan["ask"])[tuple(int(b) for b in plan["values"])].sum())
        p = torch.where(p > 0, p * torch.log2(torch.where(p > 0, p, 1.0)), 0.0)
        entropy = -float(p.sum())
        del p
        keep(psi, n, plan["collapse"], plan["values"][:1])
        at = pick(psi, first_draw(seed))
        keep(psi, n, plan["measure"], [at >> q & 1 for q in plan["measure"]])
        return {"probability": prob, "entropy": entropy, "bits": None, "state": permuted(psi, n, list(range(n)), plan["order"])}
    if kind == "batch":
        out = []
        for q, gates in small_circuits(case, rng):
            psi = zero_state(q)
            for m, t, c in gates:
                apply_gate(psi, q, m, t, c)
            out.append(psi)
        return out
    if kind == "serve":
        out = []
        for r in requests(case, rng):
            if "shots" in r:
                out.append(None)
                continue
            psi, idx = zero_state(r["n"]), torch.arange(1 << r["n"], device="cuda")
            for m, t, c in r["gates"]:
                apply_gate(psi, r["n"], m, t, c)
            out.append(torch.stack([torch.vdot(psi, apply_pauli(psi, idx, x, z)) for x, z in r["terms"]]))
        return out
    return None  # shots are whole numbers


def keep(psi, n, bits, values):
    """Only the amplitudes whose `bits` have these values, renormalised."""
    v = axes(psi, n, bits)
    for i in range(1 << len(bits)):
        at = tuple(i >> b & 1 for b in range(len(bits)))
        if at != tuple(int(b) for b in values):
            v[at].zero_()
    psi.mul_(1.0 / torch.linalg.vector_norm(torch.view_as_real(psi)))
