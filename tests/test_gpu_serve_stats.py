"""The request loop's count of launches: a request with outputs over the same request that only
returns its state."""
import pytest

from hiqsimulator_amd.circuits import random_layers_circuit
from hiqsimulator_amd.serving import make_server

pytestmark = pytest.mark.gpu


def launches(submit):
    server = make_server("c128", state_bytes=64 << 20, matrix_bytes=16 << 20)
    submit(server)
    while not server.idle():
        server.step(True)
    return server.stats()["launches"]


def test_launches_of_outputs(engine_mod):
    n = 10
    gates = random_layers_circuit(n, 4, 3)
    print("launch counts", flush=True)
    base = launches(lambda s: s.submit_state(n, gates))
    # block sums, running sums, shots
    assert launches(lambda s: s.submit_samples(n, gates, 100, 1)) == base + 3
    # eight strings a launch
    assert launches(lambda s: s.submit_expectation(n, gates, list(range(1, 18)), list(range(17)))) == base + 3
