"""Requests of very uneven shot counts that finish in one step: each one's outcomes are those it has alone."""
import numpy as np
import pytest

from hiqsimulator_amd.circuits import random_layers_circuit
from hiqsimulator_amd.serving import make_server

pytestmark = pytest.mark.gpu


def test_uneven_shots_in_one_step(engine_mod):
    shots = [1, 3, 2 ** 18, 5, 1, 1000, 4, 2, 7, 1]
    reqs = [(5 + i, random_layers_circuit(5 + i, 3, 50 + i), s, 900 + i) for i, s in enumerate(shots)]

    def serve(some):
        server = make_server("c128", state_bytes=64 << 20, matrix_bytes=16 << 20)
        ids = [server.submit_samples(*r) for r in some]
        while not server.idle():
            server.step(True)
        return [np.asarray(server.samples(i)) for i in ids]

    print("uneven shots", flush=True)
    for together, r in zip(serve(reqs), reqs):
        assert len(together) == r[2]
        assert np.array_equal(together, serve([r])[0])
