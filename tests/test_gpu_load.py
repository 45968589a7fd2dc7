"""Loads whose statistics are reduced on the device (egs_setup.hip: k_load_device, egs_ingest.hip:
k_rd_rows): the internal game, MG and values equal the host's at the edges of their tiles."""
import numpy as np
import pytest

from conftest import lfp, to_oracle_game

pytestmark = pytest.mark.gpu


def _read_order(n, seed, hub=0, wmax=50):
    rng = np.random.default_rng(seed)
    deg = rng.integers(1, 5, size=n)
    if hub:
        deg[n // 2] = hub
    rptr = np.zeros(n + 1, np.int32)
    rptr[1:] = np.cumsum(deg)
    m = int(rptr[-1])
    return (rng.integers(0, 2, size=n).astype(np.uint8), rptr, rng.integers(0, n, size=m).astype(np.int32),
            rng.integers(-wmax, wmax + 1, size=m).astype(np.int32))


# one row; a tile of 256 rows and its neighbours; a row longer than the workgroup; more tiles
# than workgroups
@pytest.mark.parametrize("n,hub", [(1, 0), (2, 0), (255, 0), (256, 300), (257, 0), (1000, 70000), (270000, 5000)])
def test_read_order_load_equals_host(oracle, n, hub):
    import egsolver_amd as E
    owner, rptr, rsucc, rw = _read_order(n, 5 + n, hub)
    want = E.games.internalise(owner, rptr, rsucc, rw)
    print(f"[gpu-case] read order n {n} m {want.m}", flush=True)
    with E.Solver(n, want.m) as s:
        n0, mg, ext = s.load_read_order(owner, rptr, rsucc, rw)
        assert (n0, mg) == (want.n0, want.mg)
        assert np.array_equal(ext, want.ext_of_int)
        ptr, succ, w = s.game()
        assert np.array_equal(ptr, want.ptr) and np.array_equal(succ, want.succ) and np.array_equal(w, want.w)
        s.prepare()
        conv, _ = s.iterate()
        assert conv and s.violations() == 0
        if want.m < 5000:
            assert np.array_equal(s.values(), lfp(oracle, to_oracle_game(want)))


def test_refused_loads_keep_the_game():
    """A game with a fault is refused with its message, and the one loaded before stays."""
    import egsolver_amd as E
    owner, rptr, rsucc, rw = _read_order(3000, 1)
    with E.Solver(3000, 20000) as s:
        s.load_read_order(owner, rptr, rsucc, rw)
        before = s.game()
        bad = rptr.copy()
        bad[7] = bad[6]
        with pytest.raises(Exception, match="no out-edge"):
            s.load_read_order(owner, bad, rsucc, rw)
        bad = rsucc.copy()
        bad[11] = 3000
        with pytest.raises(Exception, match="out of range"):
            s.load_read_order(owner, rptr, bad, rw)
        assert all(np.array_equal(a, b) for a, b in zip(before, s.game()))
        heavy = np.full_like(rw, -2147483648)
        with pytest.raises(Exception, match="overflow"):
            s.load_read_order(owner, rptr, rsucc, heavy)


@pytest.mark.parametrize("n,hi", [(1, 1), (4095, 3), (4097, 700), (300001, 6)])
def test_device_load_equals_host_load(n, hi):
    """Device arrays in: the internal game, and a solve that relies on the largest degree and
    weight found on the way."""
    import torch
    import egsolver_amd as E
    rng = np.random.default_rng(n)
    deg = rng.integers(1, hi + 1, size=n)
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(deg)
    m = int(ptr[-1])
    succ = rng.integers(0, n, size=m).astype(np.int32)
    w = rng.integers(-3, 4, size=m).astype(np.int32)
    w[m - 1] = -77                                     # the largest |w| on the last edge
    g = E.Game(n=n, n0=n // 2, ptr=ptr, succ=succ, w=w, mg=E.games.compute_mg(n, ptr, w),
               ext_of_int=np.arange(n, dtype=np.int32))
    print(f"[gpu-case] device load n {n} m {m}", flush=True)
    d = [torch.from_numpy(a).cuda() for a in (ptr, succ, w)]
    torch.cuda.synchronize()
    with E.Solver(n, m) as s, E.Solver(n, m) as ref:
        s.load_device(g.n, g.n0, g.m, g.mg, *[a.data_ptr() for a in d])
        ref.load(g)
        assert all(np.array_equal(a, b) for a, b in zip(s.game(), ref.game()))
        for x in (s, ref):
            x.prepare()
            conv, _ = x.iterate()
            assert conv
        assert np.array_equal(s.values(), ref.values())


def test_load_behind_a_queued_prepare():
    """A game loaded from the host while the prepare of the one before is still queued."""
    import egsolver_amd as E
    big = E.generate(E.GenParams(n=1300000, seed=5, deg_kind=E.games.DEG_UNIFORM, deg_lo=2, deg_hi=4, wmax=50))
    games = [E.generate(E.GenParams(n=n, seed=6, deg_kind=E.games.DEG_UNIFORM, deg_lo=2, deg_hi=9, wmax=50)) for n in (900, 450019)]
    print("[gpu-case] load behind a queued prepare", flush=True)
    with E.Solver(big.n, max(big.m, games[1].m)) as s:
        for g in games:
            s.load(big)
            s.prepare(E.options(slices=4))
            s.prepare()
            s.load(g)
            s.prepare()
            conv, _ = s.iterate()
            assert conv and s.violations() == 0
            vals = s.values()
            s.prepare(E.options(slices=1, group=2))
            conv, _ = s.iterate()
            assert conv and np.array_equal(s.values(), vals)
