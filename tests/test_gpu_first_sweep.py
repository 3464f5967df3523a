"""The first sweep of a system that the cell kernel's wide shape serves: the
dense-owner kernel runs behind it until a sweep has shown whether it has
owners.  Counts bit for bit against the CPU oracle, forces within 1e-12 of the
summed contribution lengths against its squared-distance form (the reference's
expression, also in FP64, is itself off by 2e-11 of them where triangles of
random particles are long: against 80 bits 2.1e-11 where the device is at 1.2e-13)."""
import time

import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with tb3.Engine(0) as e:
        yield e


def uniform(n, density, seed):
    box = (n / density) ** (1.0 / 3.0)
    return np.random.default_rng(seed).uniform(0.0, box, (n, 3)), np.full(3, box)


def jittered(n, seed):
    per = int(np.ceil(round(n ** (1 / 3), 9)))
    rng = np.random.default_rng(seed)
    site = rng.permutation(per ** 3)[:n]
    grid = np.stack([site % per, site // per % per, site // per ** 2], 1)
    return (grid + 0.5) * 0.8 + rng.normal(0.0, 0.05, (n, 3)), np.full(3, 0.8 * per)


def half_dense(n, seed):
    """Narrow by its mean density, its dense half past the narrow shape."""
    P, L = jittered(n, seed)
    keep = (P[:, 0] < L[0] / 2) | (np.random.default_rng(seed).random(n) < 0.2)
    return P[keep], L


@pytest.mark.parametrize("system,cutoff", [
    (lambda: uniform(4000, 2.0, 1), 2.6),   # some lists past 136: the kernel stays
    (lambda: uniform(4000, 2.0, 2), 2.45),  # none expected, none there
    (lambda: jittered(4096, 3), 2.65),      # expected, but a liquid's lists are shorter: it goes
    (lambda: half_dense(8000, 4), 2.5),     # the narrow shape asks for the wide one
    (lambda: half_dense(8000, 5), 2.7),     # and some of its lists are past 136
])
@pytest.mark.parametrize("first", ["forces", "energy", "step", "run"])
def test_first_sweeps(eng, oracle, system, cutoff, first):
    P, L = system()
    fo, _, co = oracle.forces_fast(P, cutoff=cutoff, L=L)
    S = oracle.force_scale(P, cutoff=cutoff, L=L)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=cutoff, domain_L=L, precision="fp64")
    if first == "energy":
        assert eng.energy()[1] == co
    elif first == "step":
        assert eng.step(0.0)[1] == co
    elif first == "run":
        assert list(eng.run(5, 0.0)) == [co] * 5
    for _ in range(3):
        _, f, _, cnt = eng.energy_grad()
        assert cnt == co and np.all(np.linalg.norm(f - fo, axis=1) <= 1e-12 * S)
    assert list(eng.run(3, 0.0)) == [co] * 3
    f = eng.get_particles()["f"]
    assert np.all(np.linalg.norm(f - fo, axis=1) <= 1e-12 * S)


def test_allocation_free_first_sweep(eng, oracle):
    import torch
    for P, L, cutoff in (*[(*uniform(4000, 2.0, 1), c) for c in (2.45, 2.6)], (*half_dense(8000, 5), 2.7)):
        fo, _, co = oracle.forces_fast(P, cutoff=cutoff, L=L)
        S = oracle.force_scale(P, cutoff=cutoff, L=L)
        eng.configure("p3bca", cutoff=cutoff, domain_L=L, precision="fp64")
        x = torch.tensor(P, device="cuda")
        E, G = torch.zeros((), dtype=torch.float64, device="cuda"), torch.empty_like(x)
        torch.cuda.synchronize()
        cnt = eng.energy_grad_dev_noalloc(len(P), x.data_ptr(), 1.0, E.data_ptr(), G.data_ptr(), want_count=True)
        assert cnt == co and np.all(np.linalg.norm(G.cpu().numpy() - fo, axis=1) <= 1e-12 * S)


def test_first_sweep_is_not_repeated(eng):
    """67500 particles, a sweep of ~0.8 ms that ~65 of 67500 lists outgrow: the
    first one after tb3_configure takes as long as the later ones, not twice."""
    import torch
    P, L = uniform(67500, 2.0, 7)
    x = torch.tensor(P, device="cuda")
    E, G = torch.zeros((), dtype=torch.float64, device="cuda"), torch.empty_like(x)
    torch.cuda.synchronize()

    def timed():
        t = time.perf_counter()
        eng.energy_grad_dev(len(P), x.data_ptr(), 1.0, E.data_ptr(), G.data_ptr())
        return time.perf_counter() - t

    first, later = [], []
    for k in range(8):
        eng.configure("p3bca", cutoff=2.6, domain_L=L, precision="fp64")
        t = timed()
        if k > 0:  # the very first one allocates
            first.append(t)
        later += [timed() for _ in range(3)]
    assert np.median(first) < 1.4 * np.median(later), (first, later)
