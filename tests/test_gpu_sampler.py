"""Sampler on the GPU against a plain inverse-CDF search over the state's own
probabilities, with the counter-based generator written out here: every shot's
outcome has positive probability and its interval of the running sum holds
U * total, up to the rounding of the sums.  Sizes around one block (256
amplitudes), the 64-way searches' remainders and the largest number of blocks;
states with long runs of zero amplitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def philox_uniform(shots, seed):
    m32 = np.uint64(0xFFFFFFFF)
    c = [np.arange(shots, dtype=np.uint64), np.zeros(shots, np.uint64),
         np.full(shots, 0x5A3D, np.uint64), np.zeros(shots, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return ((c[0] << np.uint64(21)) ^ c[1]).astype(np.float64) * 2.0 ** -53


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 3, 5, 6, 7, 8, 9, 13, 14, 15, 20, 24])
@pytest.mark.parametrize("kind", ["dense", "sparse", "basis"])
def test_sampler_matches_inverse_cdf(engine_mod, n, precision, kind):
    rng = np.random.default_rng(10 * n + len(kind))
    wf = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    if kind == "sparse":  # runs of zeros of every length, ends included
        wf[rng.random(1 << n) < 0.9] = 0
        wf[: (1 << n) // 3] = 0
        wf[-(1 << n) // 5:] = 0
        wf[rng.integers((1 << n) // 3, (1 << n) - (1 << n) // 5)] = 1
    elif kind == "basis":
        wf[:] = 0
        wf[rng.integers(1 << n)] = 1
    wf /= np.linalg.norm(wf)
    sim = engine_mod.SimulatorMPI(3, n, 4, precision)
    sim.allocate_qureg(list(range(n)), 0)
    sim.set_wavefunction(wf, list(range(n)))
    print("sampler n=%d %s %s" % (n, precision, kind), flush=True)
    shots, seed = 1001, (7 << 40) + n
    got = np.asarray(sim.sample(shots, seed), dtype=np.int64)
    v = wf.astype(np.complex64) if precision == "c64" else wf
    p = v.real.astype(np.float64) ** 2 + v.imag.astype(np.float64) ** 2
    cdf = np.cumsum(p)
    u = philox_uniform(shots, seed) * cdf[-1]
    eps = cdf[-1] * 2.0 ** (n - 51)  # both sums: at most 2^n roundings of 2^-53 each, and products
    assert np.all(p[got] > 0)
    assert np.all(u <= cdf[got] + eps)
    assert np.all(u >= cdf[got] - p[got] - eps)
