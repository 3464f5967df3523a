"""The bit-exact all-triplets sweep past 4096 particles, which computes every
length where it needs it instead of reading a table of them: whole force sums
of some particles (8.4 million triplets each), bit for bit."""
import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


def powers(d):
    p = [d]
    for _ in range(5):
        p.append(p[-1] * d)
    return p


def bracket(x, y, z, nu):
    """One side's bracket (AxilrodTeller.cpp:68-81), operation for operation."""
    t = -8. / (x[3] * y[2] * z[2])
    t = t - 1. / (y[4] * z[4])
    t = t + 5. * y[0] / (x[5] * z[4])
    t = t + 5. * z[0] / (x[5] * y[4])
    t = t - 1. / (x[1] * y[2] * z[4])
    t = t - 1. / (x[1] * y[4] * z[2])
    t = t - 3. / (x[3] * y[0] * z[4])
    t = t - 3. / (x[3] * y[4] * z[0])
    t = t - 5. / (x[5] * y[0] * z[2])
    t = t - 5. / (x[5] * y[2] * z[0])
    t = t + 6. / (x[3] * y[2] * z[2])
    return (3. * nu / (8. * x[0])) * t


def contributions(P, i, j, k, role, nu=1.0):
    """What the reference subtracts from i, j or k (AxilrodTeller.cpp:83-93)."""
    def length(d):
        return np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])
    a, b, c = P[j] - P[i], P[k] - P[i], P[k] - P[j]
    pa, pb, pc = (powers(length(d)) for d in (a, b, c))
    if role == 0:
        return a * bracket(pa, pb, pc, nu)[:, None] + b * bracket(pb, pa, pc, nu)[:, None]
    if role == 1:
        return a * (-bracket(pa, pb, pc, nu))[:, None] + c * bracket(pc, pb, pa, nu)[:, None]
    return b * (-bracket(pb, pa, pc, nu))[:, None] + c * (-bracket(pc, pb, pa, nu))[:, None]


def force(P, p):
    """Particle p's force: its contributions as i, j and k in loop order, one
    subtraction after another per role, then b0 + (b1 + b2)."""
    n = len(P)
    sums = []
    for role in range(3):
        acc = np.zeros((1, 3))
        rows = range(p + 1, n - 1) if role == 0 else range(0, p if role == 1 else p - 1)
        rows = np.array(rows, dtype=np.int64)
        for part in np.array_split(rows, max(1, len(rows) // 128)):
            first = [np.arange((e if role != 1 else p) + 1, p if role == 2 else n) for e in part]
            if not first:
                continue
            o = np.concatenate(first)
            e = np.repeat(part, [len(v) for v in first])
            q = np.full(len(o), p)
            i, j, k = ((q, e, o), (e, q, o), (e, o, q))[role]
            c = contributions(P, i, j, k, role)
            acc = np.add.accumulate(np.concatenate([acc, -c]), axis=0)[-1:]
        sums.append(acc[0])
    return sums[0] + (sums[1] + sums[2])


def jittered(n, seed):
    per = int(np.ceil(round(n ** (1 / 3), 9)))
    rng = np.random.default_rng(seed)
    site = rng.permutation(per ** 3)[:n]
    return (np.stack([site % per, site // per % per, site // per ** 2], 1) + 0.5) * 0.8 + rng.normal(0, 0.05, (n, 3))


def test_exact_all_triplets_without_the_pair_table(oracle):
    P = jittered(37, 1)
    *_, fo, _ = oracle.sweep(P, mode="owner")
    assert all(np.array_equal(force(P, p), fo[p]) for p in range(37))
    n = 4097  # the last group of four has one particle
    P = jittered(n, 2)
    with tb3.Engine(0) as eng:
        eng.set_particles(P)
        eng.configure("auta", precision="exact")
        assert eng.compute_forces() == n * (n - 1) * (n - 2) // 6
        f = eng.get_particles()["f"]
    for p in (0, 1, 2049, 4095, 4096):
        assert np.array_equal(f[p], force(P, p)), p
        print(f"particle {p}: the same bits", flush=True)
