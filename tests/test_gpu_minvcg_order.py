"""GPU MInvCG where a shift stops before the others need it to: the first shift
converges first (shifts in falling order, or looser stop residuals of its own),
which freezes the direction that every later step uses (minvcg.C:210-222 skips
a converged shift 0 too), and a recurrence that breaks down a few steps after a
shift converged, which leaves that shift's solution alone.  Against the oracle:
the same iteration counts, psi within 1e-10 relative a shift and the residuals to
1e-7 (relative link errors of 1e-14 move the oracle's own by 4e-14 and 1e-12)."""
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


# the step cap: 4 and less flush every step; 9 and 14 end with steps pending
@pytest.mark.parametrize("action", ["dwf", "mobius"])
@pytest.mark.parametrize("shifts,rsd", [([5.0, 0.5, 0.01], 1e-6),
                                        ([0.01, 0.5, 5.0], [1e-2, 1e-8, 1e-8]),
                                        ([0.0, 0.5, 5.0], [1e-2, 1e-8, 1e-3]),
                                        ([2.0, 0.1, 0.5], 1e-3)])
def test_first_shift_stops_first(action, shifts, rsd):
    g, o = make(action, (4, 2, 2, 6), 4)
    chi = np.random.default_rng(9).standard_normal(g.n)
    for cap in (2, 3, 4, 9, 14, 1000):
        print(f"[gpu] MInvCG {action} shifts={shifts} rsd={rsd} cap={cap}", flush=True)
        gp, gk, grs, git, _ = g.MInvCG(chi, 0.1, shifts, rsd, max_iter=cap)
        op, ok, ors, oit = o.minvcg(chi, 0.1, shifts, rsd, max_iter=cap)
        assert gk == ok and np.array_equal(git, oit)
        assert np.allclose(grs, ors, rtol=1e-7)
        for s in range(len(shifts)):
            assert np.linalg.norm(gp[s] - op[s]) <= 1e-10 * np.linalg.norm(op[s])
    g.close()


# 36864 (site, slice) pairs: the general hop kernels
@pytest.mark.parametrize("action", ["dwf", "mobius"])
def test_general_lattice(action):
    print(f"[gpu] MInvCG {action} 8x8x8x18 Ls 8", flush=True)
    g, o = make(action, (8, 8, 8, 18), 8)
    chi = np.random.default_rng(9).standard_normal(g.n)
    for shifts, rsd, cap in (([0.01, 0.3, 4.0], 1e-3, 11), ([4.0, 0.01], 1e-2, 11)):
        gp, gk, grs, git, _ = g.MInvCG(chi, 0.1, shifts, rsd, max_iter=cap)
        op, ok, ors, oit = o.minvcg(chi, 0.1, shifts, rsd, max_iter=cap)
        assert gk == ok and np.array_equal(git, oit) and np.allclose(grs, ors, rtol=1e-7)
        for s in range(len(shifts)):
            assert np.linalg.norm(gp[s] - op[s]) <= 1e-10 * np.linalg.norm(op[s])
    g.close()


@pytest.mark.parametrize("action", ["dwf", "mobius"])
def test_breakdown_after_a_shift_converged(action):
    """|chi|^2 of 1e-295 underflows within seven steps, the second shift having
    converged in the first: 0 / 0 from there on in the first shift only."""
    print(f"[gpu] MInvCG {action}: |r|^2 runs into underflow", flush=True)
    g, o = make(action, (4, 2, 2, 6), 4)
    chi = 1e-149 * np.random.default_rng(9).standard_normal(g.n)
    shifts, rsd = [300.0, 600.0], [1e-200, 1e-2]
    gp, gk, grs, git, _ = g.MInvCG(chi, 0.1, shifts, rsd, max_iter=20)
    op, ok, ors, oit = o.minvcg(chi, 0.1, shifts, rsd, max_iter=20)
    assert np.isnan(op[0]).all() and np.isfinite(op[1]).all()
    assert gk == ok and np.array_equal(git, oit) and abs(grs[1] - ors[1]) <= 1e-7 * ors[1]
    got, want = gp[1] * 1e149, op[1] * 1e149
    assert np.linalg.norm(got - want) <= 1e-10 * np.linalg.norm(want)
    g.close()
