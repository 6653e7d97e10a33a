"""GPU: DWFGPU_NS and DWFGPU_MRHS_SHAPE govern the FP64 passes of small lattices
too (the four-threads-per-pair kernels step aside), mrhs_shape() names the shape
that ran, and a shape that cannot run is refused.  Bar: 1e-13 per site."""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import BAD_ARG, DiracOpDwfGpu, DiracOpMobiusGpu, DwfGpuError
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
DIMS, LS, MASSES = (4, 4, 4, 8), 8, np.array([0.04, 0.1, 0.3])


def run(action):
    U = lat.random_gauge(DIMS, 0.3, 7)
    cls, kw = (DiracOpDwfGpu, {}) if action == "dwf" else (DiracOpMobiusGpu, {"b": 1.5, "c": 0.5})
    g = cls(U, DIMS, LS, m5=1.8, **kw)
    o = Oracle(DIMS, LS, action, m5=1.8, b=1.5, c=0.5, gauge_canonical=U)
    xs = [np.random.default_rng(j).standard_normal(g.n) for j in range(3)]
    vin, vout = g.multi_vector(3, xs), g.multi_vector(3)
    g.MatPcDagMatPc_mrhs_dev(vout, vin, MASSES, "f64")
    for j in range(3):
        want, _ = o.matpcdagmatpc(xs[j], MASSES[j])
        d = np.linalg.norm((vout.download(j) - want).reshape(-1, 24), axis=1)
        assert np.max(d / np.linalg.norm(want.reshape(-1, 24), axis=1)) < 1e-13
    return g.mrhs_shape()


def test_shapes_that_ran(monkeypatch):
    print("[gpu] shapes of the batched FP64 operator on a small lattice", flush=True)
    # 256 sites: 4 a work-group, one right-hand side each
    assert run("dwf") == (4, 1) and run("mobius") == (4, 1)
    monkeypatch.setenv("DWFGPU_NS", "16")
    assert run("mobius") == (16, 1)
    monkeypatch.setenv("DWFGPU_MRHS_SHAPE", "8,3")
    assert run("dwf") == (8, 3)
    monkeypatch.delenv("DWFGPU_NS")
    assert run("dwf") == (8, 3)
    monkeypatch.setenv("DWFGPU_MRHS_SHAPE", "8,99")
    with pytest.raises(DwfGpuError) as e:
        run("dwf")
    assert e.value.code == BAD_ARG
