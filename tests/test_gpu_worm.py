"""The worm update's record layouts and exit tables, and the diagonal update's
lookups, each against the oracle; and the work-queue launch with more walkers
than it has workgroups.

Bit-exact after every sweep (whole numbers, and the worm controller's FP64
bits): the layouts hold the same operators, so nothing may differ.  T = 8 leaves
sites with one operator or none (guards next to each other), T = 0.15 gives
chains of many 64-word buffers and worms that cross the periodic closure."""
import numpy as np
import pytest

from fixtures import (field_spins, job_bilayer, job_honeycomb, ladder_dimer, plaquette_ring,
                      square_heisenberg, trimer_ring)
from test_gpu_parity import _compare, _say

pytestmark = pytest.mark.gpu

MODELS = {
    # exit rows in LDS: one worm type, several
    "square": lambda sse: square_heisenberg(sse, 4, d=-0.3, hz=0.1).flat(),
    "honeycomb": lambda sse: job_honeycomb(sse, 0.3).flat(),
    # four exits to an entry; more than 8 thresholds (ranks by bucket)
    "ladder": lambda sse: ladder_dimer(sse, 8, 0.6).flat(),
    "bilayer": lambda sse: job_bilayer(sse, 0.2).flat(),
    # one, three and four sites to a bond; the last has entries with five exits
    "field": lambda sse: field_spins(sse, 5),
    "trimer": lambda sse: trimer_ring(sse, 7)[0],
    "plaquette": lambda sse: plaquette_ring(sse, 9)[0],
}


@pytest.mark.parametrize("records,k2_lds", [(0, 0), (1, 0), (2, 0), (3, 0), (0, 1536)])
@pytest.mark.parametrize("kind", MODELS)
def test_worm_layouts(sse_pkg, oracle_mod, kind, records, k2_lds):
    flat = MODELS[kind](sse_pkg)
    walkers = [sse_pkg.walker_desc(T=T, seed=60 + k, thermalization=4)
               for k, T in enumerate((0.15, 1.0, 8.0))]
    _say(f"worm layouts: {kind} records={records} k2_lds={k2_lds}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_WORM_RECORDS, records)
    if k2_lds:
        # the table and small walkers fit, then neither as the chains grow
        batch.set_option(sse_pkg.capi.SSE_OPT_K2_LDS, k2_lds)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    for o in oracles:
        o.init()
    _compare(batch, oracles, f"{kind} init")
    for s in range(12):
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"{kind} sweep {s}")
    batch.close()


@pytest.mark.parametrize("kind,size,T,cutoff", [
    ("square", 4, 0.3, 63), ("square", 4, 0.3, 64), ("square", 4, 0.3, 65),  # one table; ragged chunks
    ("square", 4, 0.05, 0),      # grown from nothing; over 64 draws of a chunk, chunks of one site's bonds
    ("ladder", 8, 0.1, 0),       # a table per bond type
    ("bilayer", 0, 0.1, 1000),   # vertices without a diagonal partner
    ("square", 40, 1.5, 0),      # lookups past the staging limit: read from global memory
])
def test_diagonal_update(sse_pkg, oracle_mod, kind, size, T, cutoff):
    """Diagonal update and vertex list alone, both as chunks and slot by slot
    (8): strings, draws and lists equal the oracle's after each."""
    model = {"square": lambda: square_heisenberg(sse_pkg, size, d=-0.3, hz=0.1),
             "ladder": lambda: ladder_dimer(sse_pkg, size, 0.6),
             "bilayer": lambda: job_bilayer(sse_pkg, T)}[kind]()
    flat = model.flat()
    walkers = [sse_pkg.walker_desc(T=T * f, seed=90 + k, init_opstring_cutoff=cutoff)
               for k, f in enumerate((1.0, 4.0))]
    _say(f"diagonal update: {kind} {size} T={T} cutoff={cutoff}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    for o in oracles:
        o.init()
    for s in range(10):
        batch.sweep_phases(3 if s % 4 else 11)
        for k, o in enumerate(oracles):
            assert o.sweep_phases(3) == 0
            gs, gops, gspins = batch.get_walker(k)
            os_, oops, ospins = o.state()
            assert gs["rng_counter"] == os_["rng_counter"]
            assert np.array_equal(gops, oops) and np.array_equal(gspins, ospins)
            for got, want in zip(batch.vertex_list(k), o.vertex_list()):
                assert np.array_equal(got, want)
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"sweep {s}")
    batch.close()


@pytest.mark.parametrize("call", ["run", "budgets", "noalloc"])
def test_work_queue_hands_walkers_over(sse_pkg, oracle_mod, call):
    """2600 walkers, more than the card holds workgroups (at most 8 to each of
    256 compute units), so a walker's sweeps pass between workgroups: all equal
    the one-stream launches, some the oracle.  Budgets of 0, 1, the segment
    count 16, one past it and 33."""
    n, T = 2600, 0.7
    flat = square_heisenberg(sse_pkg, 4, d=-0.3, hz=0.1).flat()
    walkers = [sse_pkg.walker_desc(T=T, seed=300 + k, thermalization=2) for k in range(n)]
    budgets = np.full(n, 5, dtype=np.int64)
    if call != "run":
        budgets = np.array([0, 1, 16, 17, 33, 2], dtype=np.int64)[np.arange(n) % 6]
    _say(f"work queue: {n} walkers, {call}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_PERSISTENT, 1)
    batch.init()
    for rep in range(2):
        if call == "run":
            batch.run(5, measure=True)
        elif call == "budgets":
            batch.run_budgets(budgets, measure=True)
        else:
            batch.run_budgets_noalloc(budgets, measure=True)
    sums, sumsq, counts = batch.accumulators_raw()
    assert np.array_equal(counts, np.maximum(2 * budgets - 2, 0))
    for k in list(range(6)) + [1300, n - 1]:
        o = oracle_mod.OracleWalker(sse_pkg.capi, flat, walkers[k])
        o.init()
        o.sweep(int(2 * budgets[k]))
        gs, gops, gspins = batch.get_walker(k)
        os_, oops, ospins = o.state()
        assert np.array_equal(gops, oops) and np.array_equal(gspins, ospins)
        for key in ("cutoff", "num_operators", "num_worms", "rng_counter", "sweeps"):
            assert gs[key] == os_[key], key
    one = sse_pkg.Batch([flat], walkers, mode=0)
    one.set_option(sse_pkg.capi.SSE_OPT_STREAMS, 1)
    one.init()
    for s in range(int(2 * budgets.max())):
        one.run(1, measure=True)
        for k in np.nonzero(2 * budgets == s + 1)[0]:
            a, b = batch.get_walker(int(k)), one.get_walker(int(k))
            assert a[0]["rng_counter"] == b[0]["rng_counter"] and np.array_equal(a[1], b[1])
            assert np.array_equal(a[2], b[2])
    if call == "run":
        for a, b in zip((sums, sumsq, counts), one.accumulators_raw()):
            assert np.array_equal(a, b)
    one.close()
    batch.close()


@pytest.mark.parametrize("kinds", [("trimer",), ("plaquette", "field", "trimer"), ("square", "trimer")])
def test_generic_work_queue(sse_pkg, oracle_mod, kinds):
    """Bonds of any site count, batches of one size and of several: the tuner's
    calls run every launch form (stream groups, the work queue at two LDS sizes)
    over the same chains, which stay the oracle's, sums included."""
    flats = [MODELS[k](sse_pkg) for k in kinds]
    walkers = [sse_pkg.walker_desc(model=k % len(flats), T=(0.3, 0.7, 1.5)[k % 3], seed=500 + k,
                                   thermalization=3) for k in range(70)]
    _say(f"generic work queue: {kinds}")
    batch = sse_pkg.Batch(flats, walkers, mode=0)
    batch.init()
    sweeps = 0
    while batch.tuning(0) is None and sweeps < 80:
        batch.run(8, measure=True)
        sweeps += 8
    assert batch.tuning(0) is not None and batch.tuning(0)["candidates_measured"] >= 3
    batch.run(6, measure=True)
    sweeps += 6
    for k in (0, 1, 2, 3, 4, 5, 69):
        o = oracle_mod.OracleWalker(sse_pkg.capi, flats[k % len(flats)], walkers[k])
        o.init()
        o.sweep(sweeps)
        gs, gops, gspins = batch.get_walker(k)
        os_, oops, ospins = o.state()
        assert np.array_equal(gops, oops) and np.array_equal(gspins, ospins)
        assert gs["rng_counter"] == os_["rng_counter"] and gs["sweeps"] == sweeps
    assert (batch.accumulators_raw()[2] == sweeps - 3).all()
    batch.close()


@pytest.mark.parametrize("cutoff", [255, 256, 257, 511, 1023])
@pytest.mark.parametrize("n_est", [1, 2, 4])
def test_measure_chunks(sse_pkg, oracle_mod, cutoff, n_est):
    """The measurement at operator strings about its 256-slot chunks, one pass of
    estimators and two: the oracle's values to 1e-12 (sums in another order)."""
    if n_est == 4:
        flat = job_honeycomb(sse_pkg, 0.5).flat()
    else:
        flat = square_heisenberg(sse_pkg, 4, measure=("magnetization", "staggered_magnetization")[:n_est]).flat()
    walkers = [sse_pkg.walker_desc(T=T, seed=700 + k, init_opstring_cutoff=cutoff)
               for k, T in enumerate((0.6, 2.0))]
    _say(f"measure chunks: cutoff={cutoff} estimators={n_est}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    for o in oracles:
        o.init()
    for s in range(4):
        batch.sweep(2)
        gm = batch.measure()
        for k, o in enumerate(oracles):
            o.sweep(2)
            assert np.allclose(gm[k], o.measure(), rtol=1e-12, atol=1e-13)
    batch.close()


@pytest.mark.parametrize("n", [546, 547])
def test_measure_returns_every_walker(sse_pkg, oracle_mod, n):
    """15 values a walker: 8190 come with the call's report, 8205 by a copy."""
    flat = square_heisenberg(sse_pkg, 4).flat()
    walkers = [sse_pkg.walker_desc(T=1.0, seed=900 + k) for k in range(n)]
    _say(f"measure of {n} walkers")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.init()
    batch.sweep(3)
    gm = batch.measure()
    assert len(gm) == n and len(gm[0]) == 15
    for k in (0, 1, n // 2, n - 1):
        o = oracle_mod.OracleWalker(sse_pkg.capi, flat, walkers[k])
        o.init()
        o.sweep(3)
        assert np.allclose(gm[k], o.measure(), rtol=1e-12, atol=1e-13)
    batch.close()


@pytest.mark.parametrize("n_walkers", [2, 600])
def test_large_walkers(sse_pkg, oracle_mod, n_walkers):
    """Records of more than 64 KB (some 10^4 operators), where each walker has a
    compute unit to itself and where three share one."""
    flat = square_heisenberg(sse_pkg, 32).flat()
    walkers = [sse_pkg.walker_desc(T=0.13 if k < 2 else 8.0, seed=40 + k, thermalization=3)
               for k in range(n_walkers)]
    _say(f"large walkers: {n_walkers}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers[:2]]
    batch.init()
    for o in oracles:
        o.init()
    for s in range(14):
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"sweep {s}")
    assert batch.get_walker(0)[0]["num_operators"] > 10500
    batch.close()
