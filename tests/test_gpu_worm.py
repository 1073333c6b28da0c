"""The worm update's record layouts and exit tables, each against the oracle.

Bit-exact after every sweep (whole numbers, and the worm controller's FP64
bits): the layouts hold the same operators, so nothing may differ.  T = 8 leaves
sites with one operator or none (guards next to each other), T = 0.15 gives
chains of many 64-word buffers and worms that cross the periodic closure."""
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
