"""Sparse rounds of games with hubs, whose predecessor lists carry the edges' weights: only
vertices that can rise are queued, and the fixpoint is the oracle's."""
import ctypes

import numpy as np
import pytest

from conftest import lfp, to_oracle_game

pytestmark = pytest.mark.gpu

# (n, degree kind, lo, hi, alpha, W): buckets of the transpose placed in LDS and, past 22,528
# edges, in memory; the widest weight that fits beside a destination, and one more (no weights)
GAMES = [(3000, 2, 1, 1500, 1.7, 50), (9000, 2, 1, 6000, 2.0, 30), (2500, 1, 12, 40, 0, 200),
         (700, 3, 0, 0, 0, 40), (1200, 2, 1, 600, 1.8, (1 << 20) - 1), (1200, 2, 1, 600, 1.8, 1 << 20)]


@pytest.mark.parametrize("i", range(len(GAMES)))
@pytest.mark.parametrize("certify_every", [0, -1])
def test_hub_queues_exact(oracle, i, certify_every):
    import egsolver_amd as E
    n, kind, lo, hi, alpha, W = GAMES[i]
    g = E.generate(E.GenParams(n=n, seed=90 + i, deg_kind=kind, deg_lo=lo, deg_hi=hi, alpha=alpha or 2.0, wmax=W))
    ref = lfp(oracle, to_oracle_game(g))
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        # sparse rounds from the first on, and as the frontier decides; most vertices hubs, few
        for opt in (dict(dense_pct=101, big_deg=8, huge_deg=40), dict(dense_pct=101, big_deg=64, huge_deg=300),
                    dict(dense_pct=30, big_deg=16, huge_deg=100)):
            print(f"[gpu-case] hubs {GAMES[i]} {opt}", flush=True)
            s.prepare(E.options(certify_every=certify_every, **opt))
            conv, st = s.iterate()
            assert conv
            vals = s.values()
            assert np.array_equal(vals, ref), (opt, np.count_nonzero(vals != ref))


@pytest.mark.parametrize("leaves", [500, 8192, 8193, 30000])
def test_one_workgroup_rounds_hand_over(leaves):
    """A value that travels up a chain, one vertex a round, then to `leaves` vertices at once
    (past the lists a workgroup keeps, they go to the round kernels), then up a second chain."""
    import egsolver_amd as E
    from egsolver_amd.games import Game
    chain = 4200                                  # past one launch's rounds
    # owner 1 everywhere: 0 a sink, 1..chain the first chain, then the leaves, then the second
    leaf0, second = 1 + chain, 1 + chain + leaves
    n = second + chain
    succ = np.zeros(n, np.int32)
    succ[1:leaf0] = np.arange(chain)
    succ[leaf0:second] = chain
    succ[second] = leaf0 + leaves // 2
    succ[second + 1:] = np.arange(second, n - 1)
    w = np.zeros(n, np.int32)
    w[1] = -5
    g = Game(n=n, n0=0, ptr=np.arange(n + 1, dtype=np.int32), succ=succ, w=w, mg=5, ext_of_int=np.arange(n, dtype=np.int32))
    ref = np.full(n, 5, np.int32)
    ref[0] = 0
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        print(f"[gpu-case] chain of {chain}, {leaves} leaves", flush=True)
        s.prepare(E.options(certify_every=-1, dense_pct=101))
        conv, st = s.iterate()
        assert conv and st.phases == 2 * chain + 1
        assert np.array_equal(s.values(), ref)


@pytest.mark.parametrize("steps", [600, 1200])
def test_hub_in_a_candidate_that_diverges(oracle, steps):
    """Proof passes that pass the divergence bound while several workgroups share a hub: each of
    them has to finish its part of the pass, or the hub's next lifts fold a part of its edges only.

    A staircase s_t (value t, reached in round t) makes g rise every round; in the proofs g keeps
    only its positive self-loop and diverges.  The hub follows g, three below it by its last edges."""
    import egsolver_amd as E
    from egsolver_amd.games import Game
    edges = 6000
    n = steps + 3                                 # hub, g, s_0 .. s_steps
    hub = np.full(edges, 1, np.int32)
    hub_w = np.zeros(edges, np.int32)
    hub_w[-100:] = 3
    stairs = np.arange(steps + 1, dtype=np.int32) + 2
    succ = np.concatenate([hub, [1], stairs, [2], stairs[:-1]]).astype(np.int32)
    w = np.concatenate([hub_w, [3], np.zeros(steps + 1), [0], np.full(steps, -1)]).astype(np.int32)
    deg = np.concatenate([[edges, steps + 2], np.ones(steps + 1)]).astype(np.int64)
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    g = Game(n=n, n0=1, ptr=ptr, succ=succ, w=w, mg=E.games.compute_mg(n, ptr, w), ext_of_int=np.arange(n, dtype=np.int32))
    ref = np.concatenate([[steps - 3, steps], np.arange(steps + 1)]).astype(np.int32)
    assert np.array_equal(lfp(oracle, to_oracle_game(g)), ref)
    stop = ctypes.c_uint32(0)
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        for k in range(6):
            print(f"[gpu-case] diverging hub, {steps} steps, run {k}", flush=True)
            # a stop flag keeps the sparse rounds out of one workgroup, where nothing is shared
            s.prepare(E.options(dense_pct=101, certify_every=2 + k, cert_max_passes=8192, stop_flag=stop))
            conv, st = s.iterate()
            assert conv and st.cert_attempts > 5
            vals = s.values()
            assert np.array_equal(vals, ref), (k, vals[:2], ref[:2])


@pytest.mark.parametrize("built", ["before", "after"])
def test_replaced_values_below_their_lift(built):
    """Sparse rounds from replaced values: a vertex far below its lift rises when a successor
    does, whatever that successor's value was, in a game with hubs."""
    import egsolver_amd as E
    from egsolver_amd.games import Game
    # owner 0: p takes the smaller of a and b; owner 1: hub (100 edges to the sink), a, b, sink
    succ = np.array([2, 3] + [4] * 100 + [4, 4, 4], np.int32)
    w = np.array([0, 0] + [0] * 100 + [-5, -4, 0], np.int32)
    ptr = np.array([0, 2, 102, 103, 104, 105], np.int32)
    g = Game(n=5, n0=1, ptr=ptr, succ=succ, w=w, mg=E.games.compute_mg(5, ptr, w), ext_of_int=np.arange(5, dtype=np.int32))
    stop = ctypes.c_uint32(0)
    with E.Solver(g.n, g.m) as s:
        s.load(g)
        print(f"[gpu-case] replaced values, transpose {built}", flush=True)
        # sparse rounds from the first on, or with the transpose asked for after the replacement
        s.prepare(E.options(certify_every=-1, big_deg=8, stop_flag=stop,
                            dense_pct=101 if built == "before" else 100))
        s.set_values(np.array([0, 0, 5, 3, 0], np.int32))
        if built == "after":
            s.csc()
        conv, _ = s.iterate()
        assert conv and s.values().tolist() == [4, 0, 5, 4, 0]
        assert s.violations() == 0
