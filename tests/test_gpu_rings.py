"""GPU: the rings of vectors that the CG solvers keep their last steps in.

With DWFGPU_RING_MB=0 (no ring: every step applied at once, the directions in
place) a solve agrees with the oracle as with a ring, and the batched one gives
the bits of the one with a ring: each of its updates rounds x in FP32 by itself
either way.  A solve gives a ring of more than 256 MiB back when it ends, and
takes none above the limit.  Bars of the iterates: FP64 1e-12, FP32 1e-5 and
int16 2e-3 of the oracle's after the same steps; 1e-11 a shift in MInvCG."""
import ctypes as C

import numpy as np
import pytest

from cps_veloc_amd import dwf
from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import BAD_ARG, CgArg, DiracOpDwfGpu, DiracOpMobiusGpu, DwfGpuError
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
BAR = {"f64": 1e-12, "f32": 1e-5, "i16": 2e-3}


def make(action, dims, ls, precision="f64", oracle=True):
    U = lat.random_gauge(dims, 0.3, 7)
    cls, kw = (DiracOpDwfGpu, {}) if action == "dwf" else (DiracOpMobiusGpu, {"b": 1.5, "c": 0.5})
    g = cls(U, dims, ls, m5=1.8, precision=precision, **kw)
    return g, (Oracle(dims, ls, action, m5=1.8, b=1.5, c=0.5, gauge_canonical=U) if oracle
               else None)


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert dwf.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("ring", ["0", None])
@pytest.mark.parametrize("action,precision", [("dwf", "f64"), ("mobius", "f64"), ("dwf", "f32"),
                                              ("mobius", "i16")])
def test_invcg(monkeypatch, action, precision, ring):
    if ring is not None:
        monkeypatch.setenv("DWFGPU_RING_MB", ring)
    # a small-lattice and (36864 pairs) a general one
    for dims, ls, mass in (((4, 2, 2, 6), 4, 0.2), ((8, 8, 8, 18), 8, 0.2)):
        g, o = make(action, dims, ls, precision)
        src = np.random.default_rng(11).standard_normal(g.n)
        for cap in (3, 6, 10) if precision != "f64" else (2, 5, 6, 12, 21):
            print(f"[gpu] InvCg ring={ring} {action} {precision} {dims} cap={cap}", flush=True)
            sol = np.zeros(g.n)
            it, _, _ = g.InvCg(sol, src, CgArg(mass, cap, 1e-15))
            xo, oit, _, _ = o.invcg(src, mass, stop_rsd=1e-15, max_iter=cap)
            assert it == oit
            assert np.linalg.norm(sol - xo) <= BAR[precision] * np.linalg.norm(xo)
        g.close()


@pytest.mark.parametrize("action", ["dwf", "mobius"])
def test_multi_shift_without_ring(monkeypatch, action):
    monkeypatch.setenv("DWFGPU_RING_MB", "0")
    g, o = make(action, (4, 2, 2, 6), 4)
    chi, shifts = np.random.default_rng(9).standard_normal(g.n), np.array([0.0, 0.5, 5.0])
    for cap in (5, 11):
        print(f"[gpu] MInvCG without a ring {action} cap={cap}", flush=True)
        gp, gk, _, git, _ = g.MInvCG(chi, 0.1, shifts, 1e-3, max_iter=cap)
        op, ok, _, oit = o.minvcg(chi, 0.1, shifts, 1e-3, max_iter=cap)
        assert gk == ok and np.array_equal(git, oit)
        for s in range(3):
            assert np.linalg.norm(gp[s] - op[s]) <= 1e-11 * np.linalg.norm(op[s])
    g.close()


@pytest.mark.parametrize("action", ["dwf", "mobius"])
@pytest.mark.parametrize("sloppy", ["f32", "i16"])
def test_batch_without_ring(monkeypatch, action, sloppy):
    dims, ls, masses = (4, 4, 4, 8), 8, np.array([0.04, 0.3, 0.1])
    monkeypatch.setenv("DWFGPU_MRHS_SHAPE", "8,3")  # one order of the sums (DWF tunes it)
    got = {}
    for ring in (None, "0"):
        if ring is not None:
            monkeypatch.setenv("DWFGPU_RING_MB", ring)
        g, _ = make(action, dims, ls, oracle=False)
        xs = [np.random.default_rng(20 + j).standard_normal(g.n) for j in range(3)]
        for eager in (False, True):
            print(f"[gpu] batch ring={ring} {action} {sloppy} eager={eager}", flush=True)
            sol, src = g.multi_vector(3), g.multi_vector(3, xs)
            it, tr, st, nrel = g.InvCgMrhs_dev(sol, src, CgArg(0.0, 5000, 1e-10), masses, sloppy,
                                               0.1, eager=eager)
            assert np.all(st == 0) and np.all(tr <= 1e-10) and np.all(nrel >= 2)
            x = [sol.download(j) for j in range(3)]
            if not got:
                got.update(it=it.copy(), nrel=nrel.copy(), x=x)
            assert np.array_equal(it, got["it"]) and np.array_equal(nrel, got["nrel"])
            assert all(np.array_equal(a, b) for a, b in zip(x, got["x"]))
            sol.free()
            src.free()
        g.close()


def test_limit_is_a_number(monkeypatch):
    monkeypatch.setenv("DWFGPU_RING_MB", "lots")
    with pytest.raises(DwfGpuError) as e:
        make("dwf", (4, 2, 2, 6), 4, oracle=False)
    assert e.value.code == BAD_ARG


def test_large_ring_is_given_back(monkeypatch):
    # 16^3x32 Ls 8 FP64: 96 MiB a vector, 960 MiB of ring
    for ring in (None, "100"):
        if ring is not None:
            monkeypatch.setenv("DWFGPU_RING_MB", ring)
        g, _ = make("dwf", (16, 16, 16, 32), 8, oracle=False)
        x, b = g.vector(), g.vector(np.random.default_rng(3).standard_normal(g.n))
        g.InvCg_dev(x, b, CgArg(0.1, 3, 1e-15))  # allocates the work vectors
        before = free_bytes()
        g.InvCg_dev(x, b, CgArg(0.1, 14, 1e-15))
        print(f"[gpu] ring={ring}: {(before - free_bytes()) / 2**20:.0f} MiB kept", flush=True)
        assert before - free_bytes() <= 256 << 20
        x.free()
        b.free()
        g.close()
