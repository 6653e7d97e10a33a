"""GPU: the batched Mobius operator, one launch per pass for all right-hand sides.

Each right-hand side of a batch gives the bits that it gives alone (the same
arithmetic per site), with its own mass, on lattices whose last work-group is
partly filled and whose work-groups do not divide over the XCDs.
"""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpMobiusGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32", "bf16", "i16"])
@pytest.mark.parametrize("dims,ls,nrhs", [((4, 2, 6, 4), 6, 3), ((6, 6, 2, 10), 10, 5),
                                          ((8, 8, 10, 12), 12, 2), ((4, 4, 4, 4), 16, 1)])
def test_batch_equals_single(dims, ls, nrhs, precision):
    op = DiracOpMobiusGpu(lat.random_gauge(dims, 0.3, 7), dims, ls, m5=1.8, b=1.5, c=0.5)
    masses = np.array([0.01, 0.3, 0.04, 0.005, 0.1][:nrhs])
    xs = [lat.to_reals(lat.gaussian_spinor((ls, int(np.prod(dims)) // 2), 11 + j))
          for j in range(nrhs)]
    vin, vout = op.multi_vector(nrhs, xs), op.multi_vector(nrhs)
    op.MatPcDagMatPc_mrhs_dev(vout, vin, masses, precision)
    for j in range(nrhs):
        one, res = op.multi_vector(1, [xs[j]]), op.multi_vector(1)
        op.MatPcDagMatPc_mrhs_dev(res, one, masses[j:j + 1], precision)
        got, want = vout.download(j), res.download(0)
        print(dims, ls, precision, j, float(np.abs(want).max()), flush=True)
        assert np.isfinite(want).all() and np.abs(want).max() > 0
        assert np.array_equal(got, want), j
