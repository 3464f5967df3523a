"""All-triplets sweeps of systems with a particle far away from the others:
its triplets are next to nothing, and those in the wrong order or with a
padding slot, which the tile kernel evaluates and scales by zero, have to stay
finite on the way."""
import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with tb3.Engine(0) as e:
        yield e


@pytest.mark.parametrize("precision,far,bar", [("fp32", 3e6, 2e-6), ("fp32", 1e8, 2e-6), ("fp64", 1e55, 1e-12)])
@pytest.mark.parametrize("n", [5, 64, 70, 129, 200])
def test_all_triplets_with_a_distant_particle(eng, oracle, n, precision, far, bar):
    """The others' forces and the energy are those without it, at the bars of
    the precisions, wherever it stands in the order and in the tiles."""
    rng = np.random.default_rng(n)
    site = rng.permutation(6 ** 3)[:n]
    P = (np.stack([site % 6, site // 6 % 6, site // 36], 1) + 0.5) * 0.8 + rng.normal(0, 0.05, (n, 3))
    for at in (0, 1, n // 2, n - 2, n - 1):
        rest = np.delete(P, at, 0)
        *_, fo, _ = oracle.sweep(rest, mode="owner")
        S = oracle.force_scale(rest)
        Eo, Es = oracle.energy(rest)[0], oracle.energy_scale(rest)
        Es = Es[0] if isinstance(Es, tuple) else Es
        Q = P.copy()
        Q[at] = (far, -far / 2, 0.0)
        eng.set_particles(Q)
        eng.configure("auta", precision=precision)
        E, f, _, cnt = eng.energy_grad()
        assert cnt == n * (n - 1) * (n - 2) // 6
        assert np.all(np.isfinite(f)) and abs(E - Eo) <= bar * Es
        assert np.all(np.linalg.norm(np.delete(f, at, 0) - fo, axis=1) <= bar * S)
        assert abs(eng.energy()[0] - Eo) <= bar * Es
