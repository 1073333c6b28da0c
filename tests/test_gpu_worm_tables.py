"""Exit tables that the other layout tests do not reach, against the oracle after
every sweep: exit rows with two worm types, lists of six exits, many bond types
with their exits in LDS and in global memory.  Which table a model gets is
checked on the CPU (test_worm_tables_cpu.py).

Bit-exact: the tables hold the same lists, so nothing may differ."""
import numpy as np
import pytest

from fixtures import plaquette_ring, trimer_ring
from test_gpu_parity import _compare, _say
from test_worm_tables_cpu import honeycomb_dz, random_bonds, trimer_split

pytestmark = pytest.mark.gpu

MODELS = {
    "honeycomb_dz": honeycomb_dz,
    "trimer_split": trimer_split,
    "random_8": lambda sse: random_bonds(sse, 8),
    "random_32": lambda sse: random_bonds(sse, 32),
}


@pytest.mark.parametrize("records", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", MODELS)
def test_exit_tables(sse_pkg, oracle_mod, kind, records):
    flat = MODELS[kind](sse_pkg)
    walkers = [sse_pkg.walker_desc(T=T, seed=160 + k, thermalization=4)
               for k, T in enumerate((0.2, 1.0, 6.0))]
    _say(f"exit tables: {kind} records={records}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_WORM_RECORDS, records)
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


@pytest.mark.parametrize("make", [trimer_ring, plaquette_ring])
@pytest.mark.parametrize("n", [7, 64])
def test_global_records_of_growing_walkers(sse_pkg, oracle_mod, make, n):
    """Global records of three- and four-site bonds while a cold walker's cutoff
    grows from 64 slots: its slab holds all partners of an entry side by side at
    first (448 slots for 64), not when 394 slots are full of operators, and again
    in the next slab."""
    flat = make(sse_pkg, n)[0]
    walkers = [sse_pkg.walker_desc(T=T, seed=260 + k, init_opstring_cutoff=64, diagonal_warmup_sweeps=0)
               for k, T in enumerate((0.01, 0.05, 2.0))]
    _say(f"global records: {make.__name__} {n}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_WORM_RECORDS, 2)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    for o in oracles:
        o.init()
    full = 0.0
    for s in range(8):
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"sweep {s}")
        sc = batch.get_walker(0)[0]
        full = max(full, sc["num_operators"] if sc["cutoff"] == 394 else 0)
    # bytes of the records with 8-byte partners against the slab's
    ns = flat.bond_n_sites
    assert 10 * (ns * full + 2 * n) > 6 * (ns * 448 + 2 * n)
    batch.close()


@pytest.mark.parametrize("make,n", [(trimer_ring, 64), (plaquette_ring, 20)])
@pytest.mark.parametrize("k2_lds", [768, 1280, 2048])
def test_codes_in_lds_without_the_records(sse_pkg, oracle_mod, make, n, k2_lds):
    """Three- and four-site bonds with LDS for the codes of some walkers and not for
    their partners, for neither of others; the walkers change sides as they grow."""
    flat = make(sse_pkg, n)[0]
    walkers = [sse_pkg.walker_desc(T=T, seed=360 + k, thermalization=4)
               for k, T in enumerate((0.2, 0.35, 0.6, 1.0, 3.0))]
    _say(f"codes in LDS: {make.__name__} {k2_lds}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_K2_LDS, k2_lds)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    for o in oracles:
        o.init()
    code = 1 if flat.bond_n_sites == 3 else 2
    hybrid = 0
    for s in range(14):
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"sweep {s}")
        for k in range(len(walkers)):
            e = flat.bond_n_sites * batch.get_walker(k)[0]["num_operators"] + 2 * n
            hybrid += code * e <= k2_lds < (code + 2) * e
    assert hybrid > 0
    batch.close()


def test_generic_work_queue_hands_walkers_over(sse_pkg, oracle_mod):
    """2600 rings of three-site bonds, more than the card holds workgroups: the
    tuner's work-queue calls cut the sweeps of a walker into tasks that other
    workgroups take over, and all chains and sums stay those of one stream."""
    n = 2600
    flat = trimer_ring(sse_pkg, 6)[0]
    walkers = [sse_pkg.walker_desc(T=0.7, seed=800 + k, thermalization=2) for k in range(n)]
    _say(f"generic work queue: {n} walkers")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    batch.init()
    sweeps = 0
    while batch.tuning(0) is None and sweeps < 80:
        batch.run(8, measure=True)
        sweeps += 8
    assert batch.tuning(0)["candidates_measured"] >= 3
    batch.run(6, measure=True)
    sweeps += 6
    one = sse_pkg.Batch([flat], walkers, mode=0)
    one.set_option(sse_pkg.capi.SSE_OPT_STREAMS, 1)
    one.init()
    one.run(sweeps, measure=True)
    for a, b in zip(batch.accumulators_raw(), one.accumulators_raw()):
        assert np.array_equal(a, b)
    for k in range(0, n, 13):
        a, b = batch.get_walker(k), one.get_walker(k)
        assert a[0]["rng_counter"] == b[0]["rng_counter"]
        assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    for k in (0, 1, n // 2, n - 1):
        o = oracle_mod.OracleWalker(sse_pkg.capi, flat, walkers[k])
        o.init()
        o.sweep(sweeps)
        a, b = batch.get_walker(k), o.state()
        assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    one.close()
    batch.close()


@pytest.mark.parametrize("k2_lds,walkers", [(19712, 8), (26880, 6), (32000, 5), (32256, 4), (32768, 4), (40192, 4), (81152, 2)])
def test_residency_report(sse_pkg, k2_lds, walkers):
    """Walkers per CU as they run: a workgroup takes its LDS + 256 in steps of 512
    bytes, out of 162816."""
    flat = trimer_ring(sse_pkg, 6)[0]
    batch = sse_pkg.Batch([flat], [sse_pkg.walker_desc(T=0.7, seed=1)], mode=0)
    batch.set_option(sse_pkg.capi.SSE_OPT_K2_LDS, k2_lds)
    assert batch.lds_bytes()[1:] == (k2_lds, walkers)
    assert walkers == min(8, 162816 // (-(-(k2_lds + 256) // 512) * 512))
    batch.close()


def test_tuner_tries_more_walkers_per_cu(sse_pkg):
    """A batch of other than two-site bonds that fills the chip has one candidate
    more than a small one: eight walkers per CU."""
    flat = trimer_ring(sse_pkg, 6)[0]
    measured = []
    for n in (200, 1400):
        batch = sse_pkg.Batch([flat], [sse_pkg.walker_desc(T=0.7, seed=k, thermalization=2) for k in range(n)], mode=0)
        batch.init()
        for _ in range(20):
            if batch.tuning(0) is None:
                batch.run(8, measure=True)
        measured.append(batch.tuning(0)["candidates_measured"])
        batch.close()
    assert measured[1] == measured[0] + 1
