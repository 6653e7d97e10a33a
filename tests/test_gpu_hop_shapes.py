"""GPU: the general hop kernels at the sites per work-group that Ls, action and
format choose (16, 32, 64), against the CPU oracle, on a lattice large enough for
every one of them whose last work-group is partly filled.  Bars: FP64 1e-13 per
site, FP32 1e-5 and int16 2e-4 of the vector, as for the other shapes."""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpDwfGpu, DiracOpMobiusGpu
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
DIMS, MASS = (14, 10, 18, 12), 0.04


@pytest.mark.parametrize("action", ["dwf", "mobius"])
@pytest.mark.parametrize("ls", [4, 6, 8, 10])
def test_operator_at_each_shape(action, ls):
    print(f"[gpu] hop shapes {action} ls={ls}", flush=True)
    U = lat.random_gauge(DIMS, 0.3, 7)
    cls, kw = (DiracOpDwfGpu, {}) if action == "dwf" else (DiracOpMobiusGpu, {"b": 1.5, "c": 0.5})
    o = Oracle(DIMS, ls, action, m5=1.8, b=1.5, c=0.5, gauge_canonical=U)
    g = cls(U, DIMS, ls, m5=1.8, **kw)
    x = np.random.default_rng(5).standard_normal(g.n)
    want, dwant = o.matpcdagmatpc(x, MASS)
    got = np.zeros(g.n)
    d = g.MatPcDagMatPc(got, x, MASS)
    a, w = got.reshape(-1, 24), want.reshape(-1, 24)
    assert np.max(np.linalg.norm(a - w, axis=1) / np.linalg.norm(w, axis=1)) < 1e-13
    assert abs(d - dwant) < 1e-13 * dwant
    g.close()
    for precision, tol in (("f32", 1e-5), ("i16", 2e-4)):
        h = cls(U, DIMS, ls, m5=1.8, precision=precision, **kw)
        h.MatPcDagMatPc(got, x, MASS)
        assert np.linalg.norm(got - want) < tol * np.linalg.norm(want), precision
        h.close()
