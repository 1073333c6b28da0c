"""Exit tables that the other layout tests do not reach, against the oracle after
every sweep: exit rows with two worm types, lists of six exits, many bond types
with their exits in LDS and in global memory.  Which table a model gets is
checked on the CPU (test_worm_tables_cpu.py).

Bit-exact: the tables hold the same lists, so nothing may differ."""
import pytest

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
