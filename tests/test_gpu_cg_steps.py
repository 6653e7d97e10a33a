"""GPU InvCg capped at a number of steps where its deferred solution updates can
go wrong (the short solves that apply every step, one step less than, exactly
and more than the pending updates, twice around the ring), converging inside a
ring, and on handles of other formats (their scaled fields take the per-site
kernels).  Bars: FP64 within 1e-12 of the oracle's iterate after the same steps
(far from convergence rounding does not grow); FP32 within 1e-5 and int16 within
2e-3 of it (five to ten operator roundings of 1e-6 and 1e-4)."""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import CgArg, DiracOpDwfGpu, DiracOpMobiusGpu
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
BAR = {"f64": 1e-12, "f32": 1e-5, "i16": 2e-3}


@pytest.mark.parametrize("action,precision", [("dwf", "f64"), ("mobius", "f64"), ("dwf", "f32"),
                                              ("mobius", "i16")])
def test_invcg_after_steps(action, precision):
    dims, ls, mass = (4, 2, 2, 6), 4, 0.2
    U = lat.random_gauge(dims, 0.3, 7)
    cls, kw = (DiracOpDwfGpu, {}) if action == "dwf" else (DiracOpMobiusGpu, {"b": 1.5, "c": 0.5})
    g = cls(U, dims, ls, m5=1.8, precision=precision, **kw)
    o = Oracle(dims, ls, action, m5=1.8, b=1.5, c=0.5, gauge_canonical=U)
    src = np.random.default_rng(11).standard_normal(g.n)
    for cap in (1, 2, 3, 5, 6, 8, 9, 10, 11, 18, 27) if precision == "f64" else (3, 6, 10):
        print(f"[gpu] InvCg {action} {precision} max_num_iter={cap}", flush=True)
        sol = np.zeros(g.n)
        it, tr, st = g.InvCg(sol, src, CgArg(mass, cap, 1e-15))
        xo, oit, otr, _ = o.invcg(src, mass, stop_rsd=1e-15, max_iter=cap)
        assert it == oit
        assert np.linalg.norm(sol - xo) <= BAR[precision] * max(np.linalg.norm(xo), 1e-300)
        if precision == "f64":
            assert abs(tr - otr) <= 1e-9 * otr
    if precision == "f64":
        for stop in (1e-2, 1e-4, 1e-6, 1e-8):
            sol = np.zeros(g.n)
            it, _, st = g.InvCg(sol, src, CgArg(mass, 1000, stop))
            xo, oit, _, _ = o.invcg(src, mass, stop_rsd=stop, max_iter=1000)
            assert st == 0 and it == oit
            assert np.linalg.norm(sol - xo) <= 1e-10 * np.linalg.norm(xo)
    g.close()
