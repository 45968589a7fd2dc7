"""Read-backs through pinned memory (egs_api.hip: read_back): the mirror of a small solve, the
small area, the two halves of the large buffer, and their order with other read-backs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ring(n, wmax=9):
    """Out-degree 2 with deterministic weights: values that differ from vertex to vertex."""
    import egsolver_amd as E
    v = np.arange(n, dtype=np.int64)
    succ = np.stack([(v + 1) % n, (v * 7 + 3) % n], 1).astype(np.int32).ravel()
    w = np.stack([(v % (2 * wmax + 1)) - wmax, (v * 5 % (2 * wmax + 1)) - wmax], 1).astype(np.int32).ravel()
    ptr = np.arange(0, 2 * n + 1, 2, dtype=np.int32)
    return E.Game(n=n, n0=n // 3, ptr=ptr, succ=succ, w=w, mg=E.games.compute_mg(n, ptr, w),
                  ext_of_int=np.arange(n, dtype=np.int32))


# the mirror (thread per vertex, one workgroup), the small area's last and first sizes past it,
# and one and more chunks of 1 MB
@pytest.mark.parametrize("n", [5, 2000, 5999, 32768, 32769, 200003, (1 << 20), (1 << 20) + 1, 2500007])
def test_values_equal_device_values(n):
    import egsolver_amd as E
    g = _ring(n)
    print(f"[gpu-case] read back n {n}", flush=True)
    pattern = ((np.arange(n, dtype=np.int64) * 2654435761) & 0x3fffffff).astype(np.int32)
    with E.Solver(n, g.m) as s:
        s.load(g)
        s.prepare(E.options(max_phases=6))
        s.iterate()
        first, win = s.values(), s.winning()
        assert np.array_equal(win, first != 2147483647)
        assert np.array_equal(s.values(), first)             # also after another read-back
        assert first.any()
        s.set_values(pattern)
        assert np.array_equal(s.values(), pattern)
        s.prepare(E.options(max_phases=6))
        assert not s.values().any()


@pytest.mark.parametrize("n", [5, 2000, 5999])
@pytest.mark.parametrize("ask", ["before", "after"])
def test_values_written_by_address(n, ask):
    """Values changed through the device address are what a read-back returns."""
    import torch
    import egsolver_amd as E
    from egsolver_amd import _native as N

    class View:
        def __init__(self, address):
            self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "strides": None, "data": (int(address), False),
                                             "version": 2}
    g = _ring(n)
    print(f"[gpu-case] values by address, n {n}", flush=True)
    with E.Solver(n, g.m) as s:
        s.load(g)
        if ask == "before":
            t = torch.as_tensor(View(N.egs().egs_solver_device_values(s.h)), device="cuda")
        s.prepare()
        s.iterate()
        if ask == "after":
            t = torch.as_tensor(View(N.egs().egs_solver_device_values(s.h)), device="cuda")
        pattern = torch.arange(n, dtype=torch.int32, device="cuda") * 3 + 1
        t.copy_(pattern)
        torch.cuda.synchronize()
        assert np.array_equal(s.values(), pattern.cpu().numpy())
