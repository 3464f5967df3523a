"""The bit-exact all-triplets sweep of few particles, a workgroup per particle
and role (up to 128)."""
import time

import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with tb3.Engine(0) as e:
        yield e


def uniform(n):
    return np.random.default_rng(n).uniform(0.0, (n / 2.0) ** (1.0 / 3.0), (n, 3))


@pytest.mark.parametrize("n", [3, 4, 6, 17, 24, 25, 64, 127, 128, 129, 131])
@pytest.mark.parametrize("algo", ["nata", "auta"])
def test_same_bits_and_counts(eng, oracle, n, algo):
    P = uniform(n)
    eng.set_particles(P)
    eng.configure(algo, precision="exact")
    *_, fo, co = oracle.sweep(P, mode="owner")
    for _ in range(2):
        assert eng.compute_forces() == co
        assert np.array_equal(eng.get_particles()["f"], fo)
    V, M = np.zeros_like(P), np.ones(n)
    eng.set_particles(P)
    g = (0.0, -9.81, 0.0)
    counts = eng.run(3, 1e-6, g)
    x, v, a, f, cs = oracle.simulate(P, V, V, M, algo, 3, 1e-6, np.array(g))
    got = eng.get_particles()
    assert list(counts) == [int(c) for c in cs]
    for key, want in (("pos", x), ("vel", v), ("acc", a), ("f", f)):
        assert np.array_equal(got[key], want), key


def test_few_particles_are_a_matter_of_launches(eng):
    """8 particles: the call takes less than the FP64 sweep's (0.8 of it; 1.25
    with the pair table's launch and the roles one after another)."""
    P = uniform(8)
    took = {}
    for precision in ("exact", "fp64"):
        eng.set_particles(P)
        eng.configure("auta", precision=precision)
        times = []
        for _ in range(120):
            start = time.perf_counter()
            eng.compute_forces()
            times.append(time.perf_counter() - start)
        took[precision] = np.median(times[20:])
    assert took["exact"] < 1.05 * took["fp64"], took
