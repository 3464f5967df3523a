"""The calls that users of this engine spend their time in, with sizes over the range they run.

listed() gives the standing cases, draw() one more of the same ranges,
prepare() the inputs and the engine a program holds before the call, run()
one pass through the public entry points, work() what that pass cannot do
without, and exact() its outputs from plain torch in 64 bits.

A case's "call" is one of
  grad    at_energy and its backward on device positions: E, dE/dx, dE/dnu
          (relaxation, fits, a force provider under torch)
  energy  at_energy alone, no gradient (line searches, Monte Carlo moves)
  sweep   Engine.energy_grad of the held particles, back on the host
  batch   the same for a batch of replicas, with the per-replica counts
  run     a program's whole simulation: particles in, steps, particles out
and its "layout" the particles:
  uniform    uniform in a box at the given density (the reference's uniform
             generator; its close pairs make long runs chaotic, so only the
             bit-exact precision runs several steps from it)
  jitter     sites of a grid of spacing 0.8 moved by N(0, 0.05), a random
             subset where the count is no cube: a liquid-like state
  clusters   Gaussian clusters, sd 1, with centres uniform in a 20^3 box
  clouds     replicas of log-uniform size, each one Gaussian cloud, sd 1.5
"""
import math

import numpy as np
import torch

from threebodymdalgorithms_amd import Engine
from threebodymdalgorithms_amd.autograd import at_energy

DT = 0.001
GRAVITY = (0.0, -9.81, 0.0)
SPACING, JITTER = 0.8, 0.05
CLUSTERS, CLUSTER_BOX = 25, 20.0
CLOUD_SD, CLOUD_MIN = 1.5, 256

# Arithmetic of one triplet: the squared-distance form (a fused multiply-add
# is two operations), and the reference's expression that the bit-exact
# precision evaluates (each division and square root one operation).
FLOPS, FLOPS_EXACT = 115, 195


def listed():
    return [
        # the smallest call: a molecule-sized system, where launches and host work are all there is
        dict(name="grad_129", call="grad", algo="p3bca", precision="fp64", layout="uniform", n=129, density=2.0,
             cutoff=2.0),
        # an energy without its gradient on an odd, ordinary size
        dict(name="energy_4999", call="energy", algo="p3bca", precision="fp64", layout="uniform", n=4999,
             density=2.0, cutoff=2.0),
        # relaxation of 8000 particles by energy and gradient (benchmarks relax8k): cutoff 2.5, few and full cells
        dict(name="relax_8000", call="grad", algo="p3bca", precision="fp64", layout="jitter", n=8000, density=0.0,
             cutoff=2.5),
        # the engine's headline system: one force sweep at N = 32768, cutoff 2
        dict(name="grad_32768", call="grad", algo="p3bca", precision="fp64", layout="uniform", n=32768,
             density=2.0, cutoff=2.0),
        # the mixed precision on the same path, a ragged size
        dict(name="grad_fp32_25001", call="grad", algo="p3bca", precision="fp32", layout="jitter", n=25001,
             density=0.0, cutoff=2.0),
        # a large system that fills the chip many times
        dict(name="grad_1048576", call="grad", algo="p3bca", precision="fp64", layout="uniform", n=1048576,
             density=2.0, cutoff=2.0),
        # a fast-path simulation: 20 steps between two looks at the particles
        dict(name="run_fp64_21952", call="run", algo="p3bca", precision="fp64", layout="jitter", n=21952,
             density=0.0, cutoff=2.0, steps=20),
        # the driver's default precision on the headline system: 10 bit-exact steps
        dict(name="run_exact_32768", call="run", algo="p3bca", precision="exact", layout="uniform", n=32768,
             density=2.0, cutoff=2.0, steps=10),
        # the driver's default algorithm and precision at the size of the reference's own test: one step of 1000
        dict(name="step_nata_1000", call="run", algo="nata", precision="exact", layout="uniform", n=1000,
             density=2.0, cutoff=0.0, steps=1),
        # every triplet of 2048 particles (benchmarks auta2048)
        dict(name="auta_2048", call="sweep", algo="auta", precision="fp64", layout="uniform", n=2048, density=2.0,
             cutoff=0.0),
        # every triplet of a clustered system in the mixed precision (benchmarks clustered16k, smaller)
        dict(name="auta_fp32_3001", call="sweep", algo="auta", precision="fp32", layout="clusters", n=3001,
             density=0.0, cutoff=0.0),
        # replicas with dense cores swept together (benchmarks batch256, fewer)
        dict(name="batch_48", call="batch", algo="p3bca", precision="fp64", layout="clouds", n=2048, density=0.0,
             cutoff=2.0, replicas=48),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the call, then its precision, its size over the whole range and its cutoff."""
    most = max(work(c)["flops"] for c in listed())
    while True:
        call = rng.choice(["grad", "grad", "energy", "run", "run", "sweep", "batch"])
        density = round(rng.uniform(1.0, 2.2), 3)
        if call in ("grad", "energy"):
            precision = rng.choice(["fp64", "fp64", "fp32"])
            layout = "jitter" if precision == "fp32" else rng.choice(["uniform", "jitter"])
            c = dict(call=call, algo="p3bca", precision=precision, layout=layout, n=_log_int(rng, 64, 600000),
                     density=density if layout == "uniform" else 0.0, cutoff=round(rng.uniform(1.5, 2.75), 3))
        elif call == "run" and rng.random() < 0.75:
            precision = rng.choice(["fp64", "exact"])
            layout = "jitter" if precision == "fp64" else "uniform"
            c = dict(call=call, algo="p3bca", precision=precision, layout=layout, n=_log_int(rng, 200, 60000),
                     density=density if layout == "uniform" else 0.0, cutoff=round(rng.uniform(1.5, 2.5), 3),
                     steps=rng.randint(2, 24))
        elif call == "run":
            c = dict(call=call, algo=rng.choice(["nata", "auta"]), precision=rng.choice(["exact", "fp64"]),
                     layout="uniform", n=_log_int(rng, 100, 1800), density=density, cutoff=0.0, steps=1)
        elif call == "sweep":
            c = dict(call=call, algo=rng.choice(["nata", "auta"]), precision=rng.choice(["fp64", "fp32"]),
                     layout=rng.choice(["uniform", "clusters"]), n=_log_int(rng, 100, 3000), density=density,
                     cutoff=0.0)
        else:
            c = dict(call=call, algo="p3bca", precision="fp64", layout="clouds", n=_log_int(rng, 512, 2048),
                     density=0.0, cutoff=round(rng.uniform(1.5, 2.2), 3), replicas=_log_int(rng, 4, 48))
        # the bit-exact precision of a mid-sized all-triplets step costs the most time per operation
        if work(c)["flops"] * (6 if c["precision"] == "exact" else 1) <= most:
            return c


# -- inputs -------------------------------------------------------------------

def _box(case):
    """Edge of the cubic box the particles fill."""
    if case["layout"] == "uniform":
        return (case["n"] / case["density"]) ** (1.0 / 3.0)
    if case["layout"] == "jitter":
        return SPACING * math.ceil(round(case["n"] ** (1.0 / 3.0), 9))
    return CLUSTER_BOX


def _cloud_sizes(case):
    """Replica sizes: log-uniform from CLOUD_MIN to n, the same for every seed."""
    u = np.random.default_rng(case["n"] + case["replicas"]).uniform(size=case["replicas"])
    return np.rint(np.exp(math.log(CLOUD_MIN) + u * math.log(case["n"] / CLOUD_MIN))).astype(int)


def _positions(case, seed):
    """The particles, (n, 3) float64 on the GPU, from the seed."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    f64 = dict(dtype=torch.float64, device="cuda", generator=gen)
    n, box = case["n"], _box(case)
    if case["layout"] == "uniform":
        return torch.rand(n, 3, **f64) * box
    if case["layout"] == "jitter":
        per = round(box / SPACING)
        site = torch.randperm(per ** 3, device="cuda", generator=gen)[:n]
        grid = torch.stack([site % per, (site // per) % per, site // (per * per)], 1).double()
        return (grid + 0.5) * SPACING + JITTER * torch.randn(n, 3, **f64)
    if case["layout"] == "clusters":
        centre = torch.rand(CLUSTERS, 3, **f64) * box
        return centre[torch.arange(n, device="cuda") % CLUSTERS] + torch.randn(n, 3, **f64)
    return CLOUD_SD * torch.randn(int(_cloud_sizes(case).sum()), 3, **f64)


def _velocities(case, seed):
    """Thermal velocities for the runs, (n, 3) on the host."""
    return np.random.default_rng(seed + 1).normal(0.0, 0.1, (case["n"], 3))


def prepare(case, seed):
    x = _positions(case, seed)
    eng = Engine(0)
    state = {"case": case, "eng": eng}
    if case["call"] in ("grad", "energy"):
        # a torch program: positions on the device, the box known
        eng.configure(case["algo"], nu=1.0, cutoff=case["cutoff"], domain_L=np.full(3, _box(case)),
                      precision=case["precision"])
        state["x"] = x.requires_grad_(case["call"] == "grad")
        state["nu"] = torch.tensor(1.0, dtype=torch.float64, device="cuda", requires_grad=case["call"] == "grad")
        return state
    state["pos"] = x.cpu().numpy()
    if case["call"] == "run":
        eng.configure(case["algo"], nu=1.0, cutoff=case["cutoff"], precision=case["precision"])
        n = case["n"]
        state["vel"], state["acc"], state["mass"] = _velocities(case, seed), np.zeros((n, 3)), np.ones(n)
        return state
    eng.set_particles(state["pos"])
    eng.configure(case["algo"], nu=1.0, cutoff=case["cutoff"], precision=case["precision"])
    if case["call"] == "batch":
        eng.batch_set(np.concatenate([[0], np.cumsum(_cloud_sizes(case))]))
    return state


def run(state):
    case, eng = state["case"], state["eng"]
    if case["call"] == "grad":
        x, nu = state["x"], state["nu"]
        x.grad = nu.grad = None
        e = at_energy(x, nu, eng)
        e.backward()
        return [e.detach(), x.grad, nu.grad]
    if case["call"] == "energy":
        with torch.no_grad():
            return [at_energy(state["x"], state["nu"], eng)]
    if case["call"] == "run":
        eng.set_particles(state["pos"], state["vel"], state["acc"], state["mass"])
        if case["steps"] == 1:
            counts = [eng.step(DT, GRAVITY)[1]]
        else:
            counts = eng.run(case["steps"], DT, GRAVITY).astype(np.int64)
        p = eng.get_particles()
        return [p["pos"], p["vel"], p["acc"], p["f"], counts]
    e, f, dnu, count = eng.energy_grad()
    if case["call"] == "batch":
        return [e, f, dnu, count, eng.batch_counts().astype(np.int64)]
    return [e, f, dnu, count]


# -- what a pass cannot do without ----------------------------------------------

def _triplets(case):
    """Expected triplets of one sweep."""
    n, c = case["n"], case["cutoff"]
    if case["layout"] == "clouds":
        # the share of triplets of three Gaussian points that are pairwise within the cutoff, by sampling
        p = np.random.default_rng(1).normal(0.0, CLOUD_SD, (3, 20000, 3))
        d = [((p[a] - p[b]) ** 2).sum(1) <= c * c for a, b in ((0, 1), (0, 2), (1, 2))]
        share = float((d[0] & d[1] & d[2]).mean())
        return share * float(sum(math.comb(int(k), 3) for k in _cloud_sizes(case)))
    every = math.comb(n, 3)
    if c <= 0:
        return float(every)
    # three points of a uniform density, pairwise within c: N density^2 / 6 times (5 pi^2 / 6) c^6
    density = n / _box(case) ** 3
    return min(float(every), n * density ** 2 / 6.0 * (5.0 * math.pi ** 2 / 6.0) * c ** 6)


def work(case):
    n = int(_cloud_sizes(case).sum()) if case["layout"] == "clouds" else case["n"]
    flop = FLOPS_EXACT if case["precision"] == "exact" else FLOPS
    if case["call"] == "run":
        # positions, velocities, accelerations and masses in; all but the masses, and the forces, out
        return {"bytes": (80 + 96) * n, "flops": flop * _triplets(case) * case["steps"]}
    if case["call"] == "energy":
        return {"bytes": 24 * n + 8, "flops": flop * _triplets(case)}
    return {"bytes": 48 * n + 16, "flops": flop * _triplets(case)}


# -- the same in plain torch, 64 bits ---------------------------------------------

def _within(a, b, L, c):
    """The periodic cutoff test of two broadcast sets of positions: min(t, L - t) per axis, no wrapping."""
    t = (a - b).abs()
    t = torch.minimum(t, L - t)
    return (t[..., 0] * t[..., 0] + t[..., 1] * t[..., 1]) + t[..., 2] * t[..., 2] <= c * c


def _candidates(x, L, c):
    """Yields (particles, their candidate partners, which of those are real), a chunk of particles at a time."""
    n = x.shape[0]
    nc = torch.floor(L / (c * (1.0 + 1e-6))).long() if c > 0 else torch.zeros(3, dtype=torch.long, device=x.device)
    every = torch.arange(n, device=x.device)
    if c <= 0 or n <= 2000 or bool((nc < 3).any()):
        step = max(1, (1 << 24) // n)
        for a in range(0, n, step):
            i = every[a:a + step]
            yield i, every.expand(len(i), n), torch.ones(len(i), n, dtype=torch.bool, device=x.device)
        return
    u = x / L
    at = torch.minimum(((u - torch.floor(u)) * nc).long(), nc - 1)
    cell = (at[:, 2] * nc[1] + at[:, 1]) * nc[0] + at[:, 0]
    order = torch.argsort(cell)
    count = torch.bincount(cell, minlength=int(nc.prod()))
    start = torch.cumsum(count, 0) - count
    widest = int(count.max())
    o = torch.arange(-1, 2, device=x.device)
    offset = torch.stack(torch.meshgrid(o, o, o, indexing="ij"), -1).reshape(27, 3)
    slot = torch.arange(widest, device=x.device)
    step = max(1, (1 << 23) // (27 * widest))
    for a in range(0, n, step):
        i = order[a:a + step]
        near = (at[i][:, None] + offset) % nc
        near = (near[..., 2] * nc[1] + near[..., 1]) * nc[0] + near[..., 0]
        real = (slot < count[near][..., None]).flatten(1)
        j = order[(start[near][..., None] + slot).clamp(max=n - 1)].flatten(1)
        yield i, j, real


def _neighbours(x, L, c):
    """Yields (particles, their partners padded to one length, which of those are real)."""
    for i, j, real in _candidates(x, L, c):
        real = real & (j != i[:, None])
        if c > 0:
            real &= _within(x[i][:, None], x[j], L, c)
            most = max(1, int(real.sum(1).max()))
            real, pick = torch.topk(real.to(torch.int8), most, dim=1)
            real, j = real.bool(), torch.gather(j, 1, pick)
        yield i, j, real


def _sweep(x, L, c, nu=1.0):
    """Energy and dE/dx: each particle's sum over the pairs of its partners that are partners of each other."""
    f = torch.zeros_like(x)
    e6 = torch.zeros((), dtype=torch.float64, device=x.device)  # six times the energy: every order of every triplet
    k = 0.375 * nu
    for i, j, real in _neighbours(x, L, c):
        m = j.shape[1]
        step = max(1, (1 << 24) // (m * m))
        for a in range(0, len(i), step):
            r, p = real[a:a + step], x[j[a:a + step]]
            d = p - x[i[a:a + step]][:, None]
            ok = r[:, :, None] & r[:, None, :] & ~torch.eye(m, dtype=torch.bool, device=x.device)
            if c > 0:
                ok &= _within(p[:, :, None], p[:, None], L, c)
            one = torch.ones((), dtype=torch.float64, device=x.device)
            u2 = (d * d).sum(-1)
            u = torch.where(ok, u2[:, :, None], one)
            v = torch.where(ok, u2[:, None, :], one)
            w = torch.where(ok, ((p[:, :, None] - p[:, None]) ** 2).sum(-1), one)
            s2 = 1.0 / (u * v * w)
            A, B, C = u + v - w, u - v + w, v + w - u
            q = A * B * C * s2
            s3 = s2 * torch.sqrt(s2)
            e6 += torch.where(ok, s3 * (nu + k * q), 0.0 * one).sum()
            du = 2.0 * s3 * s2 * ((-1.5 * nu - 2.5 * k * q) * v * w + k * (C * (A + B) - A * B))
            f[i[a:a + step]] = -(torch.where(ok, du, 0.0 * one).sum(2)[..., None] * d).sum(1)
    return e6 / 6.0, f


def _bbox(x):
    """The periodic box that the engine takes from its particles: their bounding box, 1e-4 wider on each side."""
    return ((x.max(0).values + 0.0001) - (x.min(0).values - 0.0001)).abs()


def exact(case, seed):
    x, c = _positions(case, seed), case["cutoff"]
    if case["call"] in ("grad", "energy"):
        e, f = _sweep(x, torch.full((3,), _box(case), dtype=torch.float64, device="cuda"), c)
        return [e, f, e.clone()] if case["call"] == "grad" else [e]
    if case["call"] == "sweep":
        e, f = _sweep(x, _bbox(x), c)
        return [float(e), f.cpu().numpy(), float(e), None]
    if case["call"] == "batch":
        parts = [_sweep(p, _bbox(p), c) for p in torch.split(x, _cloud_sizes(case).tolist())]
        e = float(sum(p[0] for p in parts))
        return [e, torch.cat([p[1] for p in parts]).cpu().numpy(), e, None, None]
    if case["layout"] == "uniform" and case["steps"] > 1:
        return None  # the close pairs of a uniform state make any other order of the sums part from it
    L, half = _bbox(x), 0.5 * DT * DT
    v = torch.from_numpy(_velocities(case, seed)).cuda()
    a, g = torch.zeros_like(x), torch.tensor(GRAVITY, dtype=torch.float64, device="cuda")
    for _ in range(case["steps"]):
        x = x + v * DT + a[:, :1] * half  # the x acceleration on every axis, as the reference does
        f = _sweep(x, L, c)[1]
        a = g - f
        v = v + a * (0.5 * DT)
    return [t.cpu().numpy() for t in (x, v, a, f)] + [None]
