"""Workloads of the batched SSE sweep, for timing.

Each case is a batch of walkers as a user's program builds it, thermalized
and tuned, and one pass is what such a program calls between two of its own
decisions: one Carlo step (`sweep` + `measure`), one bin of sweeps (`run`),
one budgeted call (`run_budgets`), and the reads that go with it.  The
models are those of this repository's benchmark, tests and the reference's
example job: spin-1/2 Heisenberg and XXZ squares, the spin-1 honeycomb with
single-ion anisotropy, the dimer-basis ladder (local dimension 4), and the
rings of three- and four-site bonds.

The chains are Markov chains on seeded Philox streams, so the outputs of a
pass are fixed by the seed; there is no closed form to compare them with, and
`exact` is left out of this file's answers.
"""
from __future__ import annotations

import functools
import math

import numpy as np

import __graft_entry__

sse = __graft_entry__.load_package()


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One small chain driven sweep by sweep, as Carlo's own loop does: the
        # smallest call, all launches and latency (8x8, beta = 2 is the
        # benchmark's single-walker workload).
        {"name": "carlo_1_square8_b2", "call": "carlo", "model": "square", "Lx": 8, "Ly": 8,
         "d": 0.0, "hz": 0.0, "beta": 2.0, "walkers": 1, "sweeps": 1},
        # The 16 runs of one XXZ task in a field, one Carlo step per call.
        {"name": "carlo_16_xxz12x8_b4", "call": "carlo", "model": "square", "Lx": 12, "Ly": 8,
         "d": -0.3, "hz": 0.2, "beta": 4.0, "walkers": 16, "sweeps": 1},
        # The benchmark's batched workload: one bin of ten sweeps of 4096 walkers.
        {"name": "square16_b8_4096", "call": "run", "model": "square", "Lx": 16, "Ly": 16,
         "d": 0.0, "hz": 0.0, "beta": 8.0, "walkers": 4096, "sweeps": 10},
        # An oblong lattice and an odd number of walkers, fewer than fill the card.
        {"name": "square14x10_b5_333", "call": "run", "model": "square", "Lx": 14, "Ly": 10,
         "d": 0.0, "hz": 0.0, "beta": 5.0, "walkers": 333, "sweeps": 20},
        # Few large, cold walkers (some 8000 operators each).
        {"name": "square24_b10_256", "call": "run", "model": "square", "Lx": 24, "Ly": 24,
         "d": 0.0, "hz": 0.0, "beta": 10.0, "walkers": 256, "sweeps": 4},
        # A parameter scan in one batch: XXZ squares of 8 to 24 sites a side at
        # temperatures over a factor of 32, each walker with its own budget.
        {"name": "xxz_scan_2048", "call": "budgets", "model": "scan", "Lx": 24, "Ly": 24,
         "d": 0.5, "hz": 0.1, "beta": 12.0, "walkers": 2048, "sweeps": 1},
        # The dimer-basis ladder, local dimension 4: three worm types.
        {"name": "ladder64_b10_1024", "call": "run", "model": "ladder", "Lx": 64, "Ly": 1,
         "d": 0.0, "hz": 0.0, "beta": 10.0, "walkers": 1024, "sweeps": 10},
        # The reference's example job (spin-1 honeycomb with Dz), warm: many
        # runs of one task.
        {"name": "honeycomb10_b1_512", "call": "run", "model": "honeycomb", "Lx": 10, "Ly": 10,
         "d": 0.0, "hz": 0.0, "beta": 1.0, "walkers": 512, "sweeps": 10},
        # The same job colder, on a smaller lattice: long worms.
        {"name": "honeycomb6_b3_128", "call": "run", "model": "honeycomb", "Lx": 6, "Ly": 6,
         "d": 0.0, "hz": 0.0, "beta": 3.0, "walkers": 128, "sweeps": 6},
        # Three-site bonds, the benchmark's trimer ring.
        {"name": "trimer256_b8_1024", "call": "run", "model": "trimer", "Lx": 256, "Ly": 1,
         "d": 0.0, "hz": 0.0, "beta": 8.0, "walkers": 1024, "sweeps": 8},
        # Four-site bonds.
        {"name": "plaquette64_b4_1024", "call": "run", "model": "plaquette", "Lx": 64, "Ly": 1,
         "d": 0.0, "hz": 0.0, "beta": 4.0, "walkers": 1024, "sweeps": 10},
        # Parallel tempering: 64 ladders of 8 temperatures, an exchange round
        # after every sweep.
        {"name": "tempering_square8_64x8", "call": "tempering", "model": "square", "Lx": 8,
         "Ly": 8, "d": 0.0, "hz": 0.0, "beta": 8.0, "walkers": 512, "sweeps": 20},
    ]


def draw(rng):
    """One more case of the same ranges: the model and call by kind, sizes,
    temperatures and walker counts over their logarithms, odd ones among them."""
    kind = rng.choice(["carlo", "square", "square", "cold", "scan", "ladder", "honeycomb",
                       "trimer", "plaquette", "tempering"])

    def between(lo, hi, step=1):
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return max(int(lo), int(round(v / step)) * step)

    def beta(lo, hi):
        return round(math.exp(rng.uniform(math.log(lo), math.log(hi))), 2)

    c = {"call": "run", "model": "square", "Lx": 8, "Ly": 8, "d": 0.0, "hz": 0.0, "beta": 2.0,
         "walkers": 1, "sweeps": 1}
    if kind == "carlo":
        c.update(call="carlo", Lx=between(4, 16, 2), Ly=between(4, 16, 2), beta=beta(1, 6),
                 d=rng.choice([0.0, round(rng.uniform(-0.4, 0.5), 2)]),
                 hz=rng.choice([0.0, 0.2]), walkers=between(1, 64))
    elif kind == "square":
        c.update(Lx=between(8, 18, 2), Ly=between(8, 18, 2), beta=beta(2, 9),
                 d=rng.choice([0.0, 0.0, round(rng.uniform(-0.4, 0.5), 2)]),
                 hz=rng.choice([0.0, 0.1]), walkers=between(100, 4096), sweeps=rng.randint(5, 10))
    elif kind == "cold":
        c.update(Lx=between(18, 26, 2), Ly=between(18, 26, 2), beta=beta(6, 10),
                 walkers=between(64, 256), sweeps=rng.randint(2, 4))
    elif kind == "scan":
        L = rng.choice([12, 16, 24])
        c.update(call="budgets", model="scan", Lx=L, Ly=L, d=0.5, hz=0.1, beta=beta(3, 12),
                 walkers=between(256, 2048))
    elif kind == "ladder":
        c.update(model="ladder", Lx=between(16, 96), Ly=1, beta=beta(3, 10),
                 walkers=between(100, 1024), sweeps=rng.randint(5, 10))
    elif kind == "honeycomb":
        c.update(model="honeycomb", Lx=between(4, 10, 2), Ly=between(4, 10, 2),
                 beta=beta(0.5, 2.5), walkers=between(64, 512), sweeps=rng.randint(3, 8))
    elif kind == "trimer":
        c.update(model="trimer", Lx=between(24, 256), Ly=1, beta=beta(2, 8),
                 walkers=between(100, 1024), sweeps=rng.randint(4, 8))
    elif kind == "plaquette":
        c.update(model="plaquette", Lx=between(16, 96), Ly=1, beta=beta(1.5, 6),
                 walkers=between(100, 1024), sweeps=rng.randint(4, 10))
    else:
        c.update(call="tempering", Lx=between(4, 12, 2), Ly=between(4, 12, 2), beta=beta(3, 8),
                 walkers=8 * between(4, 64), sweeps=rng.randint(5, 20))
    return c


# ---------------------------------------------------------------- the models
MEASURE = ["magnetization", "staggered_magnetization"]


@functools.lru_cache(maxsize=None)
def square(Lx, Ly, d, hz):
    return sse.MagnetModel({"lattice": {"unitcell": sse.UnitCells.square, "size": (Lx, Ly)},
                            "J": 1.0, "d": d, "hz": hz, "measure": MEASURE}).flat()


@functools.lru_cache(maxsize=None)
def honeycomb(Lx, Ly):
    return sse.MagnetModel({"lattice": {"unitcell": sse.UnitCells.honeycomb, "size": (Lx, Ly)},
                            "S": 1, "J": 1.0, "Dz": 0.005645, "measure": MEASURE}).flat()


@functools.lru_cache(maxsize=None)
def ladder(Lx, j_leg):
    return sse.ClusterModel({
        "inner_model": sse.MagnetModel, "cluster_bases": (sse.ClusterBases.dimer,),
        "lattice": {"unitcell": sse.UnitCells.ladder, "size": (Lx, 1)},
        "measure_quantum_numbers": [{"name": "", "quantum_number": 2}],
        "parameter_map": {"J": ["Jr", "Jl", "Jl"]}, "Jr": 1.0, "Jl": j_leg}).flat()


class _Magnetization:
    prefix = ""


@functools.lru_cache(maxsize=None)
def ring(n, k, J, h):
    """Spin-1/2 ring whose bonds are k consecutive sites: J S.S over the pairs
    of a bond and a field h split over the bonds of a site."""
    sz = np.diag([0.5, -0.5])
    sp = np.array([[0.0, 1.0], [0.0, 0.0]])

    def lift(op, i):
        return functools.reduce(np.kron, [op if j == i else np.eye(2) for j in range(k)])

    H = np.zeros((2 ** k, 2 ** k))
    for a in range(k):
        for b in range(a + 1, k):
            H += J * (lift(sz, a) @ lift(sz, b)
                      + 0.5 * (lift(sp, a) @ lift(sp.T, b) + lift(sp.T, a) @ lift(sp, b)))
        H -= (h / k) * lift(sz, a)
    vd = sse.VertexData((2,) * k, H)
    bonds = [sse.SSEBond(1, tuple((i + j) % n + 1 for j in range(k))) for i in range(n)]
    mval = np.tile(np.array([0.5, -0.5]), (1, n, 1))
    return sse.FlatModel(sse.SSEData([vd], bonds), [_Magnetization()], n, (np.ones((1, n)), mval))


def models_and_walkers(case, seed):
    """(models, [(model index, T)]) of a case's batch."""
    T, n = 1.0 / case["beta"], case["walkers"]
    Lx, Ly, model = case["Lx"], case["Ly"], case["model"]
    if model == "square":
        return [square(Lx, Ly, case["d"], case["hz"])], [(0, T)] * n
    if model == "honeycomb":
        return [honeycomb(Lx, Ly)], [(0, T)] * n
    if model == "trimer":
        return [ring(Lx, 3, -1.0, 0.15)], [(0, T)] * n
    if model == "plaquette":
        return [ring(Lx, 4, -0.7, 0.1)], [(0, T)] * n
    if model == "ladder":  # a scan of 16 leg couplings in [0.2, 1]
        return ([ladder(Lx, round(0.2 + 0.8 * k / 15, 4)) for k in range(16)],
                [(k % 16, T) for k in range(n)])
    # scan: L in {8, 12, 16, 24} up to Lx, eight anisotropies in [-d, d],
    # beta log-uniform over a factor of 32 up to the case's
    sizes = [L for L in (8, 12, 16, 24) if L <= Lx]
    ds = [round(case["d"] * (2 * k / 7 - 1), 4) for k in range(8)]
    models = [square(L, L, d, case["hz"]) for L in sizes for d in ds]
    rng = np.random.default_rng(seed)
    pick = rng.integers(len(models), size=n)
    betas = case["beta"] * np.exp(-rng.uniform(0.0, math.log(32.0), size=n))
    return models, [(int(m), 1.0 / float(b)) for m, b in zip(pick, betas)]


# ---------------------------------------------------------------- one case
def prepare(case, seed):
    """The batch, thermalized for a short while and with the library's launch
    forms tuned, as it stands when a program starts to take its bins."""
    models, which = models_and_walkers(case, seed)
    therm = 90
    temper = case["call"] == "tempering"
    if temper:  # 8 temperatures, geometric over a factor of 8
        which = [(0, which[0][1] * 8.0 ** ((k % 8) / 7.0)) for k in range(len(which))]
    walkers = [sse.walker_desc(model=m, T=T, seed=(seed % (1 << 40)) * 65536 + k,
                               thermalization=therm)
               for k, (m, T) in enumerate(which)]
    batch = sse.Batch(models, walkers)
    batch.init()
    state = {"case": dict(case), "batch": batch}
    if case["call"] == "budgets":
        # each walker advances until the batch's costliest has done one sweep,
        # at most 64: budgets from the expected operator count, bonds / T
        cost = np.array([models[m].n_bonds / T for m, T in which])
        state["budgets"] = np.clip(np.round(cost.max() / cost), 1, 64).astype(np.int64)
        batch.sweep(40)
        for _ in range(6):
            batch.run_budgets(state["budgets"], measure=True)
    else:
        if temper:
            batch.pt_set_ladders(np.arange(len(which)).reshape(-1, 8), seed=seed, interval=1)
        batch.sweep(therm)
        batch.run(56, measure=True)
    batch.reset_accumulators()
    return state


def snapshot(batch, walker, case):
    """One walker as a checkpoint holds it; the operator string, whose length is
    the chain's own, in the leading slots of an array that has room for it, and
    the spins likewise."""
    scalars, ops, spins = batch.get_walker(walker)
    sites = 2 * case["Lx"] * case["Ly"]
    string = np.zeros(int(10 * OPERATORS[case["model"]] * case["beta"] * sites) + 1024, np.int32)
    string[:len(ops)] = ops
    state = np.zeros(sites, np.uint8)
    state[:len(spins)] = spins
    return [scalars["cutoff"], scalars["num_operators"], int(scalars["rng_counter"]),
            scalars["sweeps"], scalars["num_worms"], string, state]


def run(state):
    case, batch = state["case"], state["batch"]
    if case["call"] == "carlo":  # Carlo.sweep! and Carlo.measure! of every run
        batch.sweep(case["sweeps"])
        return np.concatenate(batch.measure())
    if case["call"] == "budgets":
        batch.run_budgets(state["budgets"], measure=True)
    else:
        batch.run(case["sweeps"], measure=True)
    # the bin's sums, and the first and last walker as a checkpoint holds them
    sums, sumsq, counts = batch.accumulators_raw()
    wlf, wlf2, wcounts = batch.worm_fractions_raw()
    out = [sums, sumsq, counts, wlf, wlf2, wcounts, snapshot(batch, 0, case),
           snapshot(batch, len(batch.walkers) - 1, case)]
    if case["call"] == "tempering":
        order, accepted, proposed, _ = batch.pt_ladders()
        out += [order, accepted, proposed]
    return out


# Operators per site and unit of beta at low temperature, by model.
OPERATORS = {"square": 1.42, "scan": 1.42, "honeycomb": 4.1, "ladder": 1.8, "trimer": 1.44,
             "plaquette": 1.9}


def work(case):
    """Bytes of one pass: per walker and sweep the operator string of L slots is
    read and written once for the diagonal update and read once for the
    measurement, the linked vertex list (a code and one link per leg) of the n
    operators is written and read once, the W scattered vertices are rewritten, and
    the N spins pass in and out.  Operations: the 53-bit draw, weight and compare
    of every slot and the draw and exit search of every scatter, some 20 each."""
    models, which = models_and_walkers(case, 0)
    sweeps = np.full(len(which), case["sweeps"])
    betas = np.array([1.0 / T for _, T in which])
    if case["call"] == "budgets":
        cost = np.array([models[m].n_bonds / T for m, T in which])
        sweeps = np.clip(np.round(cost.max() / cost), 1, 64)
    elif case["call"] == "tempering":
        betas = betas * 8.0 ** (-(np.arange(len(which)) % 8) / 7.0)
    sites = np.array([models[m].n_sites for m, _ in which], dtype=float)
    legs = 2 * models[0].bond_n_sites
    n = OPERATORS[case["model"]] * betas * sites
    L, W = 3.0 * n, 2.0 * n
    per = 12 * L + 8 * (1 + legs) * n + 4 * W + 2 * sites
    return {"bytes": float(np.sum(per * sweeps)), "flops": float(np.sum(20 * (L + W) * sweeps))}


def exact(case, seed):
    return None
