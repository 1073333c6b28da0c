"""Diagonal update of strings whose first 64 slots hold off-diagonal operators
alone: no slot of the first chunk draws, while the random words' buffer is still
empty.  Against the oracle, bit for bit, through the two-site and the generic
kernels and through bonds of three sites."""
import numpy as np
import pytest

from fixtures import square_heisenberg, trimer_ring
from test_gpu_parity import _compare, _say

pytestmark = pytest.mark.gpu


def off_diagonal_string(flat, length, cutoff):
    """(operators, spins): on bond 0, a vertex that changes the states and the one
    that changes them back in turn, `length` times, then identities."""
    vd, ns = flat.types[int(flat.bond_type[0])], flat.bond_n_sites
    legs = np.asarray(vd["leg_states"]).reshape(vd["n_vertices"], 2 * ns)
    lower, upper = [tuple(x) for x in legs[:, :ns]], [tuple(x) for x in legs[:, ns:]]
    a = next(v for v in range(len(legs)) if lower[v] != upper[v])
    b = next(v for v in range(len(legs)) if lower[v] == upper[a] and upper[v] == lower[a])
    ops = np.zeros(cutoff, np.uint32)
    ops[:length] = [1 | (2 * v) << 1 for v in (a, b)] * (length // 2)
    spins = np.ones(flat.n_sites, np.uint8)
    spins[np.asarray(flat.bond_sites).reshape(-1, ns)[0]] = lower[a]
    return ops, spins


@pytest.mark.parametrize("kind", ["square", "generic", "trimer"])
@pytest.mark.parametrize("length", [64, 128, 254])
def test_chunk_without_draws(sse_pkg, oracle_mod, kind, length):
    flat = trimer_ring(sse_pkg, 7)[0] if kind == "trimer" else square_heisenberg(sse_pkg, 4, d=-0.3, hz=0.1).flat()
    walkers = [sse_pkg.walker_desc(T=T, seed=460 + k, init_opstring_cutoff=600) for k, T in enumerate((0.2, 2.0))]
    _say(f"chunk without draws: {kind} {length}")
    batch = sse_pkg.Batch([flat], walkers, mode=0)
    if kind == "generic":
        batch.set_option(sse_pkg.capi.SSE_OPT_GENERIC, 1)
    oracles = [oracle_mod.OracleWalker(sse_pkg.capi, flat, w) for w in walkers]
    batch.init()
    ops, spins = off_diagonal_string(flat, length, 600)
    for k, o in enumerate(oracles):
        o.init()
        sc = dict(batch.get_walker(k)[0], cutoff=len(ops), num_operators=length, num_worms=2.0)
        batch.set_walker(k, sc, ops, spins)
        assert o.set_state(sc, ops, spins) == 0
    for s in range(4):
        batch.sweep(1)
        for o in oracles:
            o.sweep(1)
        _compare(batch, oracles, f"sweep {s}")
    batch.close()
