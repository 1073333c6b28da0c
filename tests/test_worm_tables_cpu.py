"""The worm update's exit tables against the transition lists they are made
from: for every vertex, worm type and leg, and for words at and beside every
threshold, at both ends of the range and inside the tail, the exit that a table
gives is the list's first with r < cumulative probability (vertex_data.jl:113-125).
The tables are built by the library's own host code (csrc/worm_tables.h) and
looked up here as the kernels do (csrc/sse_worm.h); where a table leaves a word to
the exact search, the search is the list itself and there is nothing to compare."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from fixtures import (field_spins, job_bilayer, job_honeycomb, ladder_dimer, plaquette_ring,
                      square_heisenberg, trimer_ring)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FULL, TAIL = 1 << 53, (1 << 53) - 4096


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("worm_tables") / "libworm_tables.so")
    subprocess.run(["hipcc", "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-shared", "-w",
                    "-o", out, os.path.join(ROOT, "tests", "worm_tables_host.cpp")], check=True)
    lib = C.CDLL(out)
    lib.wt_build.restype = C.c_void_p
    lib.wt_build.argtypes = [C.c_void_p, C.POINTER(C.c_char_p)]
    lib.wt_free.argtypes = [C.c_void_p]
    lib.wt_info.argtypes = [C.c_void_p, C.POINTER(C.c_int64)]
    lib.wt_slab_bytes.restype = C.c_int64
    lib.wt_slab_bytes.argtypes = [C.c_int64, C.c_int, C.c_int, C.c_int]
    lib.wt_image.restype = C.c_void_p
    lib.wt_image.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_int64)]
    return lib


class Tables:
    def __init__(self, host, sse, flat):
        descs = sse.capi.ModelDescs([flat])
        why = C.c_char_p()
        h = host.wt_build(C.cast(descs.array, C.c_void_p), C.byref(why))
        self.refused = why.value
        if not self.refused:
            info = (C.c_int64 * 4)()
            host.wt_info(h, info)
            self.nthr, self.lg, self.mw, self.nent = info

            def image(which, dtype):
                n = C.c_int64()
                p = host.wt_image(h, which, C.byref(n))
                return np.frombuffer(C.string_at(p, n.value) if n.value else b"", dtype=dtype).copy()

            self.thr = image(0, np.uint64)
            self.row = image(1, np.uint32)
            self.exit = image(2, np.uint32).reshape(-1, 4)
            self.wide = image(3, np.uint32).reshape(self.nent, -1)
            self.code = image(4, np.uint32).reshape(-1, 2)
            self.bond = image(5, np.uint32).reshape(-1, 4)
        host.wt_free(h)
        self.ns, self.ports = flat.bond_n_sites, 2 * getattr(self, "mw", 0)

    def rank(self, m):
        return int(np.searchsorted(self.thr[:self.nthr], np.uint64(m), side="right"))

    def kind(self):
        return "rows" if len(self.row) else "exits" if len(self.exit) else "wide"

    # an exit as (selector, port, new code), or None: left to the exact search
    def rows(self, ix, m):
        w = int(self.row[self.rank(m) * self.nent + ix])
        return (w & 63) >> 4, (w >> 8) & 255, ((w >> 16) & 255) >> self.lg

    def exits(self, ix, m):
        x = [int(v) for v in self.exit[ix]]
        q = self.rank(m)
        j = sum(q >= ((x[2] >> (10 * k)) & 511) for k in range(3))
        o = ((x[0] | x[1] << 32) >> (16 * j)) & 0xFFFF
        if self.ns == 4 and q >= (x[3] & 0xFFFF):
            o = x[3] >> 16
        if m >= TAIL or o & 0x8000:
            return None
        lcb = 2 if self.ns <= 2 else 3
        return o & ((1 << lcb) - 1), (o >> lcb) & ((1 << (8 - lcb)) - 1), o >> 8

    def wides(self, ix, m):
        x, w = [int(v) for v in self.wide[ix]], m >> 21
        r, out = x[:3], x[3:7]
        if self.ns == 4:
            r, out = r + [x[7]], out + [x[8]]
        o = out[next((k for k in range(len(r)) if w < r[k]), len(r))]
        if w in r or w == 0xFFFFFFFF or o >> 31:
            return None
        step = (o >> 20) & 0x7FF
        code = (ix // self.ports) >> self.lg
        return (o & 127) >> 4, (o >> 7) & 0x1FFF, code + (step - 2048 if step >= 1024 else step)


def k_of(c):
    return 0 if c <= 0 else FULL if c >= 1 else -int(-(c * 2.0 ** 53) // 1)


def words(ks, rng):
    near = {k + d for k in ks for d in (-1 << 22, -1 << 21, -1, 0, 1, 1 << 21, 1 << 22)}
    near |= {0, 1, FULL // 2, TAIL - 1, TAIL, TAIL + 1, FULL - 2, FULL - 1}
    near |= {int(x) for x in rng.integers(0, FULL, size=8)}
    return sorted(m for m in near if 0 <= m < FULL)


def check(tab, flat):
    """Every lookup of every table of the model; returns how many a table answered."""
    ns, legs = tab.ns, 2 * tab.ns
    rng = np.random.default_rng(5)
    base = {}
    for b in range(flat.n_bonds):
        base[int(flat.bond_type[b])] = int(tab.bond[b][2])
    answered = 0
    for t, vd in enumerate(flat.types):
        if t not in base:
            continue
        off = np.asarray(vd["transition_offset"]).ravel()
        cnt = np.asarray(vd["transition_count"]).ravel()
        cum, tgt = vd["exit_cumprob"], vd["exit_target"]
        mw = vd["max_worm_count"]
        for v in range(vd["n_vertices"]):
            for wv in range(tab.mw):
                for leg in range(legs):
                    src = (v * mw + wv) * legs + leg
                    o, n = (int(off[src]), int(cnt[src])) if wv < mw else (-1, 0)
                    if o < 0:
                        n = 0
                    pos, side = leg % ns, leg // ns
                    if n == 0 and wv >= max(1, vd["dims"][pos] - 1):
                        continue  # no worm of this type lives on the site
                    ix = (((base[t] + v) << tab.lg) + pos) * tab.ports + 2 * wv + side
                    ks = [k_of(cum[o + j]) for j in range(n)]
                    for m in words(ks, rng):
                        j = next((j for j in range(n) if m < ks[j]), None)
                        want = None
                        if j is not None:
                            lo = int(vd["exit_leg"][o + j])
                            rel, up = (lo % ns + ns - pos) % ns, lo // ns
                            want = (rel | up << (1 if ns <= 2 else 2),
                                    2 * (int(vd["exit_worm"][o + j]) - 1) + (up ^ 1),
                                    base[t] + (int(tgt[o + j]) >> 1))
                        for name in ("rows", "exits", "wides"):
                            if name != "wides" and name != tab.kind():
                                continue
                            got = getattr(tab, name)(ix, m)
                            if got is not None or name == "rows":
                                assert got == want, (name, t, v, wv, leg, m)
                                answered += 1
    return answered


def honeycomb_dz(sse):
    """Spin-1 honeycomb with single-ion anisotropy: rows with two worm types."""
    return sse.MagnetModel({"lattice": {"unitcell": sse.UnitCells.honeycomb, "size": (2, 2)}, "S": 1,
                            "J": 1.0, "Dz": 0.005645, "measure": ["magnetization"]}).flat()


def with_list(flat, n, change):
    """flat with the first transition of n exits replaced: change(cumulative
    probabilities) edits them in place; None takes the transition out."""
    vd = dict(flat.types[0])
    for key in ("transition_offset", "transition_count", "exit_cumprob"):
        vd[key] = np.array(vd[key], copy=True)
    cnt = vd["transition_count"].reshape(-1)
    i = int(np.nonzero((cnt == n) & (vd["transition_offset"].reshape(-1) >= 0))[0][0])
    o = int(vd["transition_offset"].reshape(-1)[i])
    if change is None:
        vd["transition_offset"].reshape(-1)[i] = -1
    else:
        change(vd["exit_cumprob"][o:o + n])
    flat.types = [vd] + list(flat.types[1:])
    return flat


def inner_tail(c):
    c[-2], c[-1] = 1.0 - 2.0 ** -50, 1.0


def random_bonds(sse, n):
    """An XXZ square in a field whose bonds have n different anisotropies."""
    parts = [square_heisenberg(sse, 4, d=-0.3 + 0.6 * k / n, hz=0.1).flat() for k in range(n)]
    flat = parts[0]
    flat.types = [p.types[0] for p in parts]
    flat.bond_type = np.arange(flat.n_bonds) % n
    return flat


def trimer_split(sse):
    """The three-site ring with the last exit of every list of four cut in three:
    six exits with the same outcomes, beyond what an entry holds."""
    flat = trimer_ring(sse, 7)[0]
    vd = dict(flat.types[0])
    off = np.array(vd["transition_offset"]).reshape(-1)
    cnt = np.array(vd["transition_count"]).reshape(-1)
    keys = ("exit_cumprob", "exit_target", "exit_leg", "exit_worm")
    lists = {k: [] for k in keys}
    for i in range(len(off)):
        if off[i] < 0:
            continue
        part = {k: list(vd[k][off[i]:off[i] + cnt[i]]) for k in keys}
        if cnt[i] == 4:
            a, b = part["exit_cumprob"][2:4]
            for k in keys:
                part[k] = part[k][:3] + [part[k][3]] * 3
            part["exit_cumprob"][3:5] = [a + (b - a) * 0.25, a + (b - a) * 0.75]
        off[i], cnt[i] = len(lists["exit_cumprob"]), len(part["exit_cumprob"])
        for k in keys:
            lists[k] += part[k]
    vd.update({k: np.array(lists[k], dtype=np.asarray(vd[k]).dtype) for k in keys})
    vd.update(transition_offset=off, transition_count=cnt, n_exits=len(lists["exit_cumprob"]))
    flat.types = [vd]
    return flat


MODELS = {
    "square": (lambda sse: square_heisenberg(sse, 4, d=-0.3, hz=0.1).flat(), "rows"),
    "honeycomb_dz": (honeycomb_dz, "rows"),
    "field": (lambda sse: field_spins(sse, 5), None),
    "honeycomb": (lambda sse: job_honeycomb(sse, 0.3).flat(), "exits"),
    "ladder": (lambda sse: ladder_dimer(sse, 8, 0.6).flat(), "exits"),
    "bilayer": (lambda sse: job_bilayer(sse, 0.2).flat(), None),
    "trimer": (lambda sse: trimer_ring(sse, 7)[0], "exits"),
    "plaquette": (lambda sse: plaquette_ring(sse, 9)[0], "exits"),
    "trimer_split": (trimer_split, "exits"),
    "random_8": (lambda sse: random_bonds(sse, 8), "exits"),
    "random_32": (lambda sse: random_bonds(sse, 32), "wide"),
}


@pytest.mark.parametrize("name", MODELS)
def test_tables_are_the_lists(sse_pkg, host, name):
    make, kind = MODELS[name]
    flat = make(sse_pkg)
    tab = Tables(host, sse_pkg, flat)
    assert not tab.refused
    if kind:
        assert tab.kind() == kind
    assert check(tab, flat) > 0


@pytest.mark.parametrize("name,n", [("square", 2), ("honeycomb_dz", 3)])
def test_inner_threshold_in_the_tail(sse_pkg, host, name, n):
    """An exit of probability 2^-50 behind the others: words past its threshold
    lie in the tail that exit rows do not look up exactly."""
    flat = with_list(MODELS[name][0](sse_pkg), n, inner_tail)
    check(Tables(host, sse_pkg, flat), flat)


@pytest.mark.parametrize("name", ["square", "honeycomb_dz"])
def test_missing_transition(sse_pkg, host, name):
    """A vertex and leg without a transition list: the worm that gets there is an
    error of the chain, which the exact search reports; no table may answer."""
    for n in (1, 2, 3):
        flat = MODELS[name][0](sse_pkg)
        if (np.asarray(flat.types[0]["transition_count"]) == n).any():
            flat = with_list(flat, n, None)
            check(Tables(host, sse_pkg, flat), flat)


def test_bond_type_without_a_worm_type(sse_pkg, host):
    """Two bond types of one vertex whose worms only bounce, on spin-1 sites that
    hold two worm types; the second knows one.  The other worm's arrival there is
    an error as well."""
    flat = square_heisenberg(sse_pkg, 4).flat()

    def bounce(mw):
        n = mw * 4
        return dict(flat.types[0], dims=(3, 3), n_vertices=1, leg_states=np.ones((1, 4), np.uint8),
                    weights=np.ones(1), signs=np.ones(1, np.int8), diagonal_vertices=-np.ones(9, np.int32),
                    max_worm_count=mw, transition_offset=np.arange(n), transition_count=np.ones(n, np.int32),
                    n_exits=n, exit_cumprob=np.ones(n), exit_target=np.ones(n, np.int32),
                    exit_leg=np.arange(n) % 4, exit_worm=np.arange(n) // 4 + 1)

    flat.types = [bounce(2), bounce(1)]
    flat.bond_type = np.arange(flat.n_bonds) % 2
    flat.site_dims = np.full(flat.n_sites, 3, np.uint8)
    check(Tables(host, sse_pkg, flat), flat)
    flat.types = [bounce(2), bounce(2)]
    tab = Tables(host, sse_pkg, flat)
    assert tab.kind() == "rows" and check(tab, flat) > 0


@pytest.mark.parametrize("name", ["honeycomb", "ladder", "trimer", "plaquette"])
def test_word_of_a_missing_exit(sse_pkg, host, name):
    """The step loads the entry and table word behind an exit before it sees that
    there is none: the missing exit's word has to name a leg and a port that exist."""
    flat = MODELS[name][0](sse_pkg)
    tab = Tables(host, sse_pkg, flat)
    assert tab.kind() == "exits"
    lcb = 2 if tab.ns <= 2 else 3
    words = np.concatenate([tab.exit[:, 0] & 0xFFFF, tab.exit[:, 0] >> 16, tab.exit[:, 1] & 0xFFFF,
                            tab.exit[:, 1] >> 16] + ([tab.exit[:, 3] >> 16] if tab.ns == 4 else []))
    none = words[(words & 0x8000) != 0]
    assert len(none)
    assert ((none & ((1 << (lcb - 1)) - 1)) < tab.ns).all()
    assert ((none >> lcb & ((1 << (8 - lcb)) - 1)) < tab.ports).all()


@pytest.mark.parametrize("cap", [64, 448, 100032])
@pytest.mark.parametrize("sites", [16, 64, 2304])
def test_serving_footprint(host, cap, sites):
    """Admission by memory counts what the slab pool hands out: the guards of the
    batch's largest lattice come with every slab."""
    from importlib import import_module
    sv = import_module("sse_amd.serving")
    assert sv.slab_bytes(cap, sites) == host.wt_slab_bytes(cap, 2, 6, sites)
    assert sv.footprint_bytes(sites, 128, 1.0) == sv.slab_bytes(898, sites)
