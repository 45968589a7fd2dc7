"""Binned dense rounds (egs_bins.h): equal to sweeps in place at the sizes where the rule, the
slices and the chunks begin and end, for every weight range, and through the entry points that
take a game over part-way."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOP = 2147483647


def _say(msg):
    print(f"[gpu-case] {msg}", flush=True)


def _generate(n, kind, lo, hi, alpha, wmax, seed):
    import egsolver_amd as E
    return E.generate(E.GenParams(n=n, seed=seed, deg_kind=kind, deg_lo=lo, deg_hi=hi, alpha=alpha, wmax=wmax))


def _sweeps(s, **opt):
    """The loaded game by sweeps in place: an explicit slice count keeps them."""
    import egsolver_amd as E
    s.prepare(E.options(slices=1, **opt))
    conv, _ = s.iterate()
    assert conv and s.violations() == 0
    return s.values()


# (n, degree kind, lo, hi, alpha, W): below and at the least size; below and at the least average
# degree; hubs across many chunks; the largest weights of a packed word and past them; MG where
# the closure's headroom (mg + 2 W < 2^31 - 1) ends; half slices up to 2^21 vertices and whole
# ones above, where a thinner average degree is enough
GAMES = [(399999, 0, 4, 4, 0, 100), (400000, 0, 4, 4, 0, 100), (400001, 1, 2, 5, 0, 50), (450007, 2, 1, 50000, 2.1, 100),
         (524288, 2, 1, 400000, 1.8, 30), (400003, 0, 4, 4, 0, 5300), (420001, 0, 5, 5, 0, 65535), (420001, 0, 5, 5, 0, 65536),
         (1 << 21, 0, 4, 4, 0, 100), ((1 << 21) + 1, 0, 4, 4, 0, 100), ((1 << 21) + 1, 1, 3, 4, 0, 100), (2500009, 2, 1, 90000, 2.2, 40)]


@pytest.mark.parametrize("i", range(len(GAMES)))
def test_binned_rounds_exact(i):
    import egsolver_amd as E
    n, kind, lo, hi, alpha, wmax = GAMES[i]
    if wmax > 5300:                     # MG within 31 bits: heavy edges on a few vertices only
        g = _generate(n, kind, lo, hi, alpha, 3, 60 + i)
        w = g.w.copy()
        for v in range(0, n, n // 64):
            w[g.ptr[v]] = wmax if v % 2 else -wmax
        mg = E.games.compute_mg(g.n, g.ptr, w)
        g = E.Game(n=g.n, n0=g.n0, ptr=g.ptr, succ=g.succ, w=w, mg=mg, ext_of_int=g.ext_of_int)
    else:
        g = _generate(n, kind, lo, hi, alpha, wmax, 60 + i)
    _say(f"binned n {g.n} m {g.m} maxdeg {g.max_outdeg} mg {g.mg}")
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        want = _sweeps(s)
        # proofs of two passes at most would leave a skewed game to climb to MG round by round
        short = {"cert_max_passes": 64 if kind == 2 else 2}
        for opt in ({}, {"certify_every": 2}, {"certify_every": 3, **short}, {"dense_pct": 1}):
            _say(str(opt))
            s.prepare(E.options(**opt))
            assert not s.values().any()
            conv, st = s.iterate()
            assert conv and st.converged
            vals = s.values()
            assert np.array_equal(vals, want), (opt, np.count_nonzero(vals != want))
            assert s.violations() == 0
        conv, again = s.iterate()       # a converged run stays as it is
        assert conv and np.array_equal(s.values(), want)


@pytest.mark.parametrize("at", [0, 1, 3])
def test_one_vertex_holds_most_edges(at):
    """A vertex with 600,000 edges, over a hundred chunks: first, last of owner 0, last of all."""
    import egsolver_amd as E
    n, hub = 400009, 600000
    n0 = n // 2
    rng = np.random.default_rng(5 + at)
    v = {0: 0, 1: n0 - 1, 3: n - 1}[at]
    deg = np.full(n, 2, np.int64)
    deg[v] = hub
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(deg)
    m = int(ptr[-1])
    succ = rng.integers(0, n, m).astype(np.int32)
    w = rng.integers(-3, 4, m).astype(np.int32)
    g = E.Game(n=n, n0=n0, ptr=ptr, succ=succ, w=w, mg=E.games.compute_mg(n, ptr, w), ext_of_int=np.arange(n, dtype=np.int32))
    _say(f"hub at {v}, m {m}")
    with E.Solver(n, m) as s:
        s.load(g)
        # a bounded number of rounds: binned rounds are synchronous, so their values are those
        # of the rounds computed here
        s.prepare(E.options(certify_every=-1))
        conv, st = s.iterate(4)
        assert st.phases == 4
        vals = np.zeros(n, np.int64)
        src = np.repeat(np.arange(n), deg)
        for _ in range(4):
            a = vals[succ]
            c = np.where(a == TOP, TOP, np.maximum(a - w, 0))
            c[c > g.mg] = TOP
            lo = np.full(n, TOP, np.int64)
            hi = np.zeros(n, np.int64)
            np.minimum.at(lo, src, c)
            np.maximum.at(hi, src, c)
            new = np.where(np.arange(n) < n0, lo, hi)
            lifted = int(np.count_nonzero(new > vals))
            vals = np.maximum(vals, new)
        assert np.array_equal(s.values(), vals)
        assert lifted <= st.lifted


@pytest.mark.parametrize("kind,hi,alpha", [(1, 8, 0), (2, 60000, 2.1)])
def test_taken_over_part_way(kind, hi, alpha):
    """Capped runs and their resumption, the transpose before and after, replaced values, the
    certificate of the TOP set, captured rounds, and a load after a half-run game."""
    import egsolver_amd as E
    from egsolver_amd import verify
    g = _generate(410009, kind, 2 if kind == 1 else 1, hi, alpha, 100, 9)
    other = _generate(400100, 1, 2, 8, 0, 20, 10)
    _say(f"taken over n {g.n} m {g.m}")
    with E.Solver(g.n, max(g.m, other.m)) as s:
        s.load(g)
        want = _sweeps(s)
        s.prepare()
        for cap in (0, 1, 2, 5):
            conv, st = s.iterate(max_phases=cap)
            assert not conv and np.all(s.values() <= want)
        assert st.phases == 8 and st.initial_active > 0
        conv, st = s.iterate()
        assert conv and np.array_equal(s.values(), want)
        s.prepare(E.options(max_phases=4))
        conv, st = s.iterate()
        assert not conv and st.phases == 4
        s.prepare()
        cptr, _ = s.csc()                           # before the first round
        assert cptr[-1] == g.m
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), want)
        s.prepare()
        s.iterate(max_phases=3)
        s.csc()                                     # part-way
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), want)
        s.prepare()
        s.set_values(want)
        assert s.violations() == 0
        assert np.array_equal(s.values(), want)
        rep = verify.certify(s, g, want)
        assert rep["ok"], rep
        s.prepare(E.options(graphs=1))
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), want)
        stop = ctypes.c_uint32(0)
        s.prepare(E.options(stop_flag=stop))
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), want)
        s.prepare()
        s.iterate(max_phases=3)
        s.load(other)
        a = _sweeps(s)
        s.prepare()
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), a)


def test_no_initial_lift():
    """Weights without a negative edge: nothing is active, and the run ends at zero."""
    import egsolver_amd as E
    g = _generate(400010, 0, 4, 4, 0, 10, 3)
    g = E.Game(n=g.n, n0=g.n0, ptr=g.ptr, succ=g.succ, w=np.abs(g.w), mg=E.games.compute_mg(g.n, g.ptr, np.abs(g.w)),
               ext_of_int=g.ext_of_int)
    _say("no initial lift")
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        s.prepare()
        conv, st = s.iterate()
        assert conv and st.phases == 0 and st.initial_active == 0
        assert not s.values().any() and s.violations() == 0


def test_stop_flag_before_the_first_round():
    """A run stopped before it begins does no round, the one done with the layout included; with
    the flag cleared it goes on to the fixpoint."""
    import egsolver_amd as E
    g = _generate(410009, 1, 2, 8, 0, 100, 9)
    _say("stopped before the first round")
    stop = ctypes.c_uint32(1)
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        want = _sweeps(s)
        s.prepare(E.options(stop_flag=stop))
        conv, st = s.iterate()
        assert not conv and st.phases == 0 and st.lifted == 0 and st.initial_active > 0
        assert not s.values().any()
        stop.value = 0
        conv, st = s.iterate()
        assert conv and np.array_equal(s.values(), want)


@pytest.mark.parametrize("extra", [0, 1, 2, 3])
def test_any_edge_capacity(extra):
    """The vertex numbers lie behind the packed words, whose room follows from the capacity."""
    import egsolver_amd as E
    g = _generate(400013, 1, 2, 8, 0, 100, 12)
    _say(f"capacity m + {extra}")
    with E.Solver(g.n, g.m + extra) as s:
        s.load(g)
        want = _sweeps(s)
        s.prepare()
        conv, _ = s.iterate()
        assert conv and np.array_equal(s.values(), want)


def test_solver_where_memory_is_short():
    """A solver whose full work space does not fit the free memory goes without the binned layout
    and the transpose's weights, and solves large uniform and skewed games all the same."""
    import torch
    import egsolver_amd as E
    games = [_generate(430007, 1, 2, 8, 0, 100, 9), _generate(450007, 2, 1, 50000, 2.1, 100, 63)]
    n_cap, m_cap = 1 << 20, 1 << 29
    want = []
    for g in games:
        with E.Solver(g.n, g.m) as s:
            s.load(g)
            want.append(_sweeps(s))
    torch.cuda.empty_cache()
    free0 = torch.cuda.mem_get_info()[0]
    with E.Solver(n_cap, m_cap):
        full = free0 - torch.cuda.mem_get_info()[0]
    assert full > 40 * m_cap
    left = int(0.75 * full)
    _say(f"full {full >> 20} MiB, left {left >> 20} MiB")
    held, step = [], 32 << 30
    try:
        while (over := torch.cuda.mem_get_info()[0] - left) > 1 << 20:
            held.append(torch.empty(min(step, over), dtype=torch.uint8, device="cuda"))
        with E.Solver(n_cap, m_cap) as s:
            for g, w in zip(games, want):
                s.load(g)
                for opt in ({}, {"dense_pct": 60}):
                    s.prepare(E.options(**opt))
                    conv, _ = s.iterate()
                    assert conv and np.array_equal(s.values(), w)
    finally:
        held.clear()
        torch.cuda.empty_cache()
