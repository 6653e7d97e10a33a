"""GPU MInvCG where its deferred updates can go wrong: solves that end inside,
at and after a flush of pending steps (8), the short solves that flush every
step (up to 4 steps), shifts that converge early, one shift and the most (32),
no operator shift, and the SINGLE sum, against the oracle after the same number
of steps.  Bar: 1e-11 relative a shift (FP64 recurrences of the same steps, far
from convergence, differ by rounding only) and the same iteration counts."""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpDwfGpu, DiracOpMobiusGpu
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def make(action, dims, ls):
    U = lat.random_gauge(dims, 0.3, 7)
    cls, kw = (DiracOpDwfGpu, {}) if action == "dwf" else (DiracOpMobiusGpu, {"b": 1.5, "c": 0.5})
    g = cls(U, dims, ls, m5=1.8, **kw)
    return g, Oracle(dims, ls, action, m5=1.8, b=1.5, c=0.5, gauge_canonical=U)


@pytest.mark.parametrize("action,nshift,first", [("dwf", 1, 0.01), ("dwf", 32, 0.01),
                                                 ("mobius", 3, 0.0), ("mobius", 5, 0.02)])
@pytest.mark.parametrize("steps", [1, 2, 4, 5, 7, 8, 9, 10, 17])
def test_after_steps(action, nshift, first, steps):
    print(f"[gpu] MInvCG {action} nshift={nshift} steps={steps}", flush=True)
    g, o = make(action, (4, 2, 2, 6), 4)
    chi = np.random.default_rng(9).standard_normal(g.n)
    shifts = first + np.linspace(0.0, 1.0, nshift) ** 2 * 20.0
    gp, gk, grs, git, gst = g.MInvCG(chi, 0.1, shifts, 1e-3, max_iter=steps)
    op, ok, ors, oit = o.minvcg(chi, 0.1, shifts, 1e-3, max_iter=steps)
    assert gk == ok and np.array_equal(git, oit)
    assert np.allclose(grs, ors, rtol=1e-9)
    for s in range(nshift):
        assert np.linalg.norm(gp[s] - op[s]) <= 1e-11 * np.linalg.norm(op[s])
    alpha, start = np.cos(np.arange(nshift)), np.roll(chi, 24)
    sp, sk, _, _, _ = g.MInvCG(chi, 0.1, shifts, 1e-3, multi=False, alpha=alpha, psi=start,
                               max_iter=steps)
    want = start + sum(a * p for a, p in zip(alpha, op))
    assert sk == ok and np.linalg.norm(sp - want) <= 1e-11 * np.linalg.norm(want)
    g.close()
