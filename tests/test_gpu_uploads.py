"""Uploads of two handles from two threads, of arrays long enough for the ring of
pinned buffers (which one of them gets): the exact values arrive."""
import threading

import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpDwfGpu

pytestmark = pytest.mark.gpu


def test_two_threads():
    print("[gpu] 75 MB uploads of two handles from two threads", flush=True)
    dims, ls = (16, 16, 16, 16), 12
    ops = [DiracOpDwfGpu(lat.unit_gauge(dims), dims, ls, m5=1.8) for _ in range(2)]
    vs = [o.vector() for o in ops]
    ok = [0, 0]

    def run(k):
        for q in range(4):
            x = np.random.default_rng(10 * k + q).standard_normal(ops[k].n)
            vs[k].upload(x)
            ok[k] += np.array_equal(vs[k].download(), x)

    ts = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [4, 4]
