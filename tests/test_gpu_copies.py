"""Copies between device vectors and host arrays at the sizes where the chunked
path starts, has a short last chunk, wraps its ring of buffers and is used by
two threads at once: the exact values come back."""
import threading

import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpDwfGpu

pytestmark = pytest.mark.gpu


def make(dims, ls):
    return DiracOpDwfGpu(lat.unit_gauge(dims), dims, ls, m5=1.8)


# 3.9 MB (plain copy), 4.4 MB, 14.7 MB and 75.5 MB (chunked both ways)
@pytest.mark.parametrize("dims,ls", [((8, 8, 8, 10), 8), ((4, 10, 6, 12), 16), ((10, 8, 12, 20), 8),
                                     ((16, 16, 16, 16), 12)])
def test_round_trip(dims, ls):
    print(f"[gpu] vector round trip {dims} ls={ls}", flush=True)
    op = make(dims, ls)
    x = np.random.default_rng(3).standard_normal(op.n)
    v = op.vector(x)
    assert np.array_equal(v.download(), x)
    v.upload(-x)
    assert np.array_equal(v.download(), -x)
    a, b = op.fermion_from_canonical(np.concatenate([x, 2.0 * x]))
    assert np.array_equal(op.fermion_to_canonical(a, b), np.concatenate([x, 2.0 * x]))
    op.close()


def test_two_threads():
    print("[gpu] downloads of two handles from two threads", flush=True)
    ops = [make((8, 8, 8, 16), 12) for _ in range(2)]
    xs = [np.random.default_rng(k).standard_normal(o.n) for k, o in enumerate(ops)]
    vs = [o.vector(x) for o, x in zip(ops, xs)]
    ok = [0, 0]

    def run(k):
        for _ in range(8):
            ok[k] += np.array_equal(vs[k].download(), xs[k])

    ts = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [8, 8]
