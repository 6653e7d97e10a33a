"""GPU: the network's weights on the device (k_ptc_weights).

The weights that training leaves give the same network, bit for bit, as the same
weights handed over with ptc_set_weights (their bf16 forms agree in every layer
and place).  From zero moments Adam's first step is lr g / (|g| + 1e-8): each
real moves by at most lr, and by lr to FP32 rounding of the weight where its
gradient is not tiny (|g| > 1e-5: the quotient is within 1e-3 of 1).
"""
import numpy as np
import pytest

from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpMobiusGpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ls", [4, 8, 12, 16])
def test_adam_step_and_forms(ls):
    dims, lr = (4, 4, 4, 4), 1e-3
    U = lat.random_gauge(dims, 0.3, 5)
    op = DiracOpMobiusGpu(U, dims, ls, m5=1.8, b=1.5, c=0.5)
    op.ptc_init(3)
    w0 = op.ptc_get_weights().copy()
    x = lat.to_reals(lat.gaussian_spinor((ls, 128), 2))
    z0 = op.ptc_apply(x)
    _, _, used = op.ptc_train(0.04, nsolves=1, pairs_per_solve=0, random_pairs=3, epochs=1,
                              batch=3, lr=lr, seed=9)
    assert used == 3
    w1 = op.ptc_get_weights().copy()
    step = (w1 - w0).view(np.float32)
    print(ls, "largest step / lr", np.abs(step).max() / lr, flush=True)
    assert np.abs(step).max() <= lr * (1 + 1e-3)
    assert np.mean(np.abs(np.abs(step) - lr) < 2e-3 * lr) > 0.9
    z1 = op.ptc_apply(x)
    assert not np.array_equal(z0, z1)
    other = DiracOpMobiusGpu(U, dims, ls, m5=1.8, b=1.5, c=0.5)
    other.ptc_init(4)
    other.ptc_set_weights(w1)
    assert np.array_equal(other.ptc_apply(x), z1)
    assert np.array_equal(other.ptc_get_weights(), w1)
