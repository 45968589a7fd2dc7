"""Sparse rounds of games with hubs, whose predecessor lists carry the edges' weights: only
vertices that can rise are queued, and the fixpoint is the oracle's."""
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
