"""GPU Moebius operator and a few CG steps at Ls whose M5^-1 column is swept
through LDS (no register form: 14, 18, 20), on a small and on a general FP64
lattice, against the CPU oracle.  Bars: 1e-13 per site; 1e-12 after six steps."""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import CgArg, DiracOpMobiusGpu
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,ls", [((4, 2, 6, 4), 14), ((4, 2, 2, 6), 20), ((8, 6, 10, 12), 14),
                                     ((8, 6, 10, 12), 18)])
def test_columns_through_lds(dims, ls):
    print(f"[gpu] Moebius {dims} ls={ls}", flush=True)
    U = lat.random_gauge(dims, 0.3, 7)
    g = DiracOpMobiusGpu(U, dims, ls, m5=1.8, b=1.5, c=0.5)
    o = Oracle(dims, ls, "mobius", m5=1.8, b=1.5, c=0.5, gauge_canonical=U)
    x, got = np.random.default_rng(5).standard_normal(g.n), np.zeros(g.n)
    for dag in (0, 1):
        (g.MatPcDag if dag else g.MatPc)(got, x, 0.04)
        want = o.matpc(x, 0.04, dag)
        d = np.linalg.norm((got - want).reshape(-1, 24), axis=1)
        assert np.max(d / np.linalg.norm(want.reshape(-1, 24), axis=1)) < 1e-13
    sol = np.zeros(g.n)
    it, _, _ = g.InvCg(sol, x, CgArg(0.2, 6, 1e-14))
    xo, oit, _, _ = o.invcg(x, 0.2, stop_rsd=1e-14, max_iter=6)
    assert it == oit and np.linalg.norm(sol - xo) < 1e-12 * np.linalg.norm(xo)
    g.close()
