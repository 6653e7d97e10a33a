"""GPU: ptc_init's random weights are std::normal_distribution's sequence over
std::mt19937_64, bit for bit, on top of its diagonal."""
import subprocess

import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpMobiusGpu

pytestmark = pytest.mark.gpu
NORMALS = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
int main(int, char** v) {
  std::mt19937_64 rng(strtoull(v[1], nullptr, 10));
  std::normal_distribution<double> nd(0.0, 1.0);
  for (long k = atol(v[2]); k > 0; --k) {
    const double x = nd(rng);
    fwrite(&x, sizeof x, 1, stdout);
  }
}
"""


@pytest.mark.parametrize("ls,seed", [(4, 1), (8, 20260)])
def test_sequence(tmp_path, ls, seed):
    print(f"[gpu] ptc_init ls={ls} seed={seed}", flush=True)
    src, exe = tmp_path / "normals.cpp", tmp_path / "normals"
    src.write_text(NORMALS)
    subprocess.run(["g++", "-O1", str(src), "-o", str(exe)], check=True)
    dims, scale = (4, 4, 4, 4), 0.02
    op = DiracOpMobiusGpu(lat.unit_gauge(dims), dims, ls, m5=1.8, b=1.5, c=0.5)
    op.ptc_init(seed, scale)
    w = op.ptc_get_weights()
    raw = subprocess.run([str(exe), str(seed), str(2 * w.size)], check=True, timeout=60,
                         capture_output=True).stdout
    want = (scale * np.frombuffer(raw)).astype(np.float32).view(np.complex64).copy()
    at = 0
    for cin, cout, diag in ((ls, 16, 1.0), (16, 16, 1.0), (16, ls, 0.5)):
        layer = want[at:at + 9 * cout * cin * 16].reshape(9, cout, cin, 4, 4)
        for o in range(min(cin, cout)):
            for a in range(4):
                layer[0, o, o, a, a] += np.complex64(diag)
        at += layer.size
    assert at == w.size and np.array_equal(w, want)
