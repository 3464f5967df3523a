"""The sweep kernels at the sizes where their splits and tiles have edges,
against the CPU oracle: counts bit for bit, forces and energy against the
sums' own scales (each particle's summed contribution lengths S_p, and the
energy's summed magnitudes), at the bars of the precisions: 1e-12 in FP64,
2e-6 (forces) and 1e-6 (energy) in FP32-mixed."""
import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu

BARS = {"fp64": (1e-12, 1e-12), "fp32": (2e-6, 1e-6)}


def jittered(n, seed, spacing=0.8, sd=0.05):
    """n random sites of a cubic grid, each moved by N(0, sd)."""
    per = int(np.ceil(round(n ** (1 / 3), 9)))
    rng = np.random.default_rng(seed)
    site = rng.permutation(per ** 3)[:n]
    grid = np.stack([site % per, site // per % per, site // per ** 2], 1)
    return (grid + 0.5) * spacing + rng.normal(0.0, sd, (n, 3))


@pytest.fixture(scope="module")
def eng():
    with tb3.Engine(0) as e:
        yield e


def check(eng, oracle, P, precision, cutoff=-1.0, L=None):
    E, f, dnu, cnt = eng.energy_grad()
    *_, fo, co = oracle.sweep(P, cutoff=cutoff, L=L, mode="owner")
    Eo = oracle.energy(P, cutoff=cutoff, L=L)
    Eo = Eo[0] if isinstance(Eo, tuple) else Eo
    Es = oracle.energy_scale(P, cutoff=cutoff, L=L)
    Es = Es[0] if isinstance(Es, tuple) else Es
    S = oracle.force_scale(P, cutoff=cutoff, L=L)
    bar_f, bar_e = BARS[precision]
    assert cnt == co
    assert np.all(np.linalg.norm(f - fo, axis=1) <= bar_f * S)
    assert abs(E - Eo) <= bar_e * Es and dnu == E
    E2, cnt2 = eng.energy()
    assert cnt2 == co and abs(E2 - Eo) <= bar_e * Es


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [3, 4, 63, 64, 65, 127, 128, 129, 193, 450])
def test_all_triplets_tile_edges(eng, oracle, n, precision):
    P = jittered(n, n)
    eng.set_particles(P)
    eng.configure("auta", precision=precision)
    check(eng, oracle, P, precision)


@pytest.mark.parametrize("n", [3, 4, 5, 8, 9, 65, 130, 257, 699, 702])
def test_exact_all_triplets_group_edges(eng, oracle, n):
    """Bit for bit at the edges of the bit-exact sweep's rounds (64 items and
    multiples) and particle groups (2 below 700 particles, 4 from there)."""
    P = jittered(n, 1000 + n)
    eng.set_particles(P)
    eng.configure("nata", precision="exact")
    assert eng.compute_forces() == n * (n - 1) * (n - 2) // 6
    *_, fo, _ = oracle.sweep(P, mode="owner")
    assert np.array_equal(eng.get_particles()["f"], fo)


def test_exact_all_triplets_out_of_range_side(eng, oracle):
    """Sides out of the in-range sequences' range: the same bits."""
    P = jittered(70, 5)
    P[0] = (1e14, 0.0, 0.0)
    eng.set_particles(P)
    eng.configure("auta", precision="exact")
    eng.compute_forces()
    *_, fo, _ = oracle.sweep(P, mode="owner")
    assert np.array_equal(eng.get_particles()["f"], fo)


def test_exact_all_triplets_past_the_pair_table(eng):
    """More particles than the table of pair lengths holds: against the FP64
    path, at the bar of the all-triplets sweep of 2048 particles."""
    n = 4100
    P = jittered(n, 6)
    eng.set_particles(P)
    eng.configure("auta", precision="exact")
    cnt = eng.compute_forces()
    f = eng.get_particles()["f"]
    eng.configure("auta", precision="fp64")
    assert cnt == eng.compute_forces() == n * (n - 1) * (n - 2) // 6
    f64 = eng.get_particles()["f"]
    size = np.linalg.norm(f, axis=1)
    floor = np.sqrt(np.mean(size ** 2))
    assert np.all(np.linalg.norm(f64 - f, axis=1) <= 2e-11 * np.maximum(size, floor))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,cutoff", [(5, 2.0), (129, 2.0), (400, 2.0), (500, 2.0), (1100, 2.0), (1728, 2.5),
                                      (3375, 2.0), (3375, 2.5), (8000, 2.0)])
def test_cutoff_cell_shapes(eng, oracle, n, cutoff, precision):
    """One to 343 cells, so that a cell's owners are split among 16 down to 3
    workgroups, in the narrow and (cutoff 2.5, or everything in one cell) the
    wide shape of the cell kernel."""
    P = jittered(n, 2000 + n)
    L = np.full(3, 0.8 * np.ceil(round(n ** (1 / 3), 9)))
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=cutoff, domain_L=L, precision=precision)
    check(eng, oracle, P, precision, cutoff=cutoff, L=L)


def test_cutoff_wide_shape_found_by_the_sweep(eng, oracle):
    """A system whose mean density asks for the narrow shape but whose dense
    half needs the wide one: the pass is repeated, and a run goes on in it."""
    rng = np.random.default_rng(11)
    P = jittered(8000, 12)
    keep = (P[:, 0] < 8.0) | (rng.random(8000) < 0.2)
    P = P[keep]
    L = np.full(3, 16.0)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=2.5, domain_L=L, precision="fp64")
    check(eng, oracle, P, "fp64", cutoff=2.5, L=L)
    eng.set_particles(P)
    counts = eng.run(3, 1e-4)
    eng.set_particles(P)
    assert [eng.step(1e-4)[1] for _ in range(3)] == [int(c) for c in counts]


def test_single_passes_share_the_slots(eng, oracle):
    """Single passes leave the slot counts ready for the next one: sweeps of
    changing particle counts, with steps, a run, a non-finite position and a
    crowded cell (more particles than slots) between them, each against the
    oracle's count of the same positions."""
    L = np.full(3, 0.8 * 12)
    eng.set_particles(jittered(1700, 30))
    eng.configure("p3bca", cutoff=2.0, domain_L=L, precision="fp64")
    rng = np.random.default_rng(31)
    crowded = np.concatenate([jittered(1500, 32), rng.uniform(4.1, 4.9, (60, 3))])
    lost = jittered(300, 33)
    lost[7] = np.nan
    for P in (jittered(1700, 30), jittered(800, 34), crowded, jittered(1728, 35), lost, jittered(900, 36), crowded):
        eng.set_particles(P)
        *_, co = oracle.sweep(P, cutoff=2.0, L=L, mode="owner")
        assert eng.compute_forces() == co
        assert eng.energy()[1] == co
        f = eng.get_particles()["f"]
        assert eng.energy_grad()[3] == co
        if np.all(np.isfinite(P)):
            S = oracle.force_scale(P, cutoff=2.0, L=L)
            assert np.all(np.linalg.norm(eng.get_particles()["f"] - f, axis=1) <= 1e-12 * S)
        eng.set_particles(P)
        assert eng.step(0.0)[1] == co
        if np.all(np.isfinite(P)):
            assert list(eng.run(3, 0.0)) == [co] * 3


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [300, 520, 900])
def test_dense_owner_lists(eng, oracle, n, precision):
    """Lists of the dense-owner kernel of one up to 15 blocks of r, even and
    odd lengths: n sites of a grid with spacing 0.8 scaled by 0.3, so that
    (almost) all are within the cutoff of each other, in a box of 5 cells
    that leaves the pair tests plain, and in one whose periodic images count."""
    P = 0.3 * jittered(n, 3000 + n)
    for box, shift in ((20.0, 10.0), (6.6, 5.8)):
        Q = P + shift
        L = np.full(3, box)
        eng.set_particles(Q)
        eng.configure("p3bca", cutoff=2.0, domain_L=L, precision=precision)
        check(eng, oracle, Q, precision, cutoff=2.0, L=L)


@pytest.mark.parametrize("n,spacing", [(4, 0.8), (30, 0.8), (300, 0.8), (700, 0.5), (1400, 0.34), (1400, 0.27)])
def test_exact_cutoff_list_lengths(eng, oracle, n, spacing):
    """Bit for bit with lists of a few entries up to past 1024, where they
    stop holding the sides to the owner (33, 65, 130, 270, ~800, ~1300
    neighbours), so that every sort and both forms of the list run."""
    P = jittered(n, 4000 + n, spacing=spacing, sd=0.06 * spacing)
    L = np.full(3, 12.0)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=2.0, domain_L=L, precision="exact")
    cnt = eng.compute_forces()
    *_, fo, co = oracle.sweep(P, cutoff=2.0, L=L, mode="owner")
    assert cnt == co
    assert np.array_equal(eng.get_particles()["f"], fo)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [4913, 5832, 9261, 12167])
def test_cutoff_heaviest_cells_split(eng, oracle, n, precision):
    """1331 to 2744 cells, a sixteenth of them split among two workgroups,
    and 3375, none of them."""
    P = jittered(n, 5000 + n, sd=0.1)
    L = np.full(3, 0.8 * round(n ** (1 / 3)))
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=1.2, domain_L=L, precision=precision)
    check(eng, oracle, P, precision, cutoff=1.2, L=L)


@pytest.mark.parametrize("n", [300, 800, 1500])
def test_cutoff_uneven_cells(eng, oracle, n):
    """A cloud in a box of 1728 cells, most of them empty: the few that hold it
    are split by their work, estimated in the first pass and measured in the
    next ones, and (n = 1500) hand owners on, one by one and cell by cell."""
    P = np.random.default_rng(n).normal(12.0, 2.0, (n, 3))
    L = np.full(3, 24.5)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=2.0, domain_L=L, precision="fp64")
    for _ in range(3):
        check(eng, oracle, P, "fp64", cutoff=2.0, L=L)


@pytest.mark.parametrize("crowded", [False, True])
def test_cutoff_large_grid_slots(eng, oracle, crowded):
    """9261 cells, past those of the fused scan: single passes fill the slots
    there too, and go back to the contiguous list where a cell outgrows them."""
    n = 42875
    P = jittered(n, 77, sd=0.1)
    if crowded:
        P[:40] = 7.0 + np.random.default_rng(78).uniform(0.0, 1.2, (40, 3))
    L = np.full(3, 28.0)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=1.3, domain_L=L, precision="fp64")
    for _ in range(2):
        check(eng, oracle, P, "fp64", cutoff=1.3, L=L)


@pytest.mark.parametrize("n", [1, 4096, 4097])
def test_particles_through_the_stage(eng, oracle, n):
    """Up to 4096 particles and the forces of a sweep pass through pinned
    memory, more through copies: the same bits come back."""
    rng = np.random.default_rng(n)
    P = jittered(n, 6000 + n) if n > 1 else np.full((1, 3), 0.4)
    V, A, M = rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.uniform(1, 2, n)
    eng.set_particles(P, V, A, M, ids=np.arange(n)[::-1])
    L = np.full(3, 0.8 * np.ceil(round(n ** (1 / 3), 9)))
    eng.configure("p3bca", cutoff=1.5, domain_L=L, precision="fp64")
    S = oracle.force_scale(P, cutoff=1.5, L=L)
    _, f, _, _ = eng.energy_grad()
    got = eng.get_particles()
    for key, want in (("pos", P), ("vel", V), ("acc", A), ("mass", M), ("id", np.arange(n)[::-1])):
        assert np.array_equal(got[key], want), key
    assert np.array_equal(got["f"], f)
    *_, fo, _ = oracle.sweep(P, cutoff=1.5, L=L, mode="owner")
    assert (np.abs(f - fo) <= 1e-12 * np.maximum(S, 1e-300)[:, None]).all()


def test_batch_after_single_passes(eng, oracle):
    """A single pass leaves the status clear, but not the sums of replicas that
    are split off after it: each replica's first counts and energies are those
    of the replica alone."""
    reps = [jittered(n, 7000 + n, sd=0.1) for n in (40, 3, 150, 9)]
    P = np.concatenate(reps)
    for first in range(2):  # the second batch meets the first one's tables
        eng.set_particles(P)
        eng.configure("p3bca", cutoff=1.7, precision="fp64")
        eng.energy_grad()
        eng.batch_set(np.concatenate([[0], np.cumsum([len(r) for r in reps])]))
        if first == 0:
            _, f, _, total = eng.energy_grad()
            counts = eng.batch_counts()
        else:
            E, counts = eng.batch_energy()
            assert float(E.sum()) == pytest.approx(alone_E, rel=1e-10)
        alone, alone_E = [], 0.0
        for r in reps:
            eng.set_particles(r)
            e, _, _, c = eng.energy_grad()
            alone.append(c)
            alone_E += e
        assert [int(c) for c in counts] == alone
        if first == 0:
            assert total == sum(alone)


@pytest.mark.parametrize("nu", ["number", "host tensor", "device tensor"])
def test_energy_waits_for_the_positions(eng, nu):
    """Positions that torch's default stream is still about to write: the
    energy is that of the written ones, wherever nu's value lives."""
    import torch
    from threebodymdalgorithms_amd.autograd import at_energy
    P, Q = jittered(500, 1), jittered(500, 2)
    eng.set_particles(P)
    eng.configure("p3bca", cutoff=2.0, domain_L=np.full(3, 6.4), precision="fp64")
    x, q = torch.tensor(P, device="cuda"), torch.tensor(Q, device="cuda")
    nus = {"number": 1.0, "host tensor": torch.tensor(1.0, dtype=torch.float64),
           "device tensor": torch.tensor(1.0, dtype=torch.float64, device="cuda")}
    want = float(at_energy(q, 1.0, eng))
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    for _ in range(20):
        a = a @ a * 1e-2
    x.copy_(q)
    with torch.no_grad():
        got = at_energy(x, nus[nu], eng)
    assert float(got) == pytest.approx(want, rel=1e-10)
