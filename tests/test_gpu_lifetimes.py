"""GPU: vectors outlive their operator.  Closing the operator first (Python
drops its objects in any order) leaves them valid to free, and their device
memory comes back."""
import ctypes as C

import pytest

from cps_veloc_amd import dwf
from cps_veloc_amd import lattice as lat
from cps_veloc_amd.dwf import DiracOpDwfGpu

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert dwf.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_vectors_freed_after_the_operator():
    print("[gpu] vectors freed after their operator", flush=True)
    dims, ls = (8, 8, 8, 16), 8
    for _ in range(2):  # the second round starts from warm pools
        before = free_bytes()
        op = DiracOpDwfGpu(lat.unit_gauge(dims), dims, ls, m5=1.8)
        one, many = op.vector(), op.multi_vector(12)
        op.close()
        other = DiracOpDwfGpu(lat.unit_gauge((4, 4, 4, 4)), (4, 4, 4, 4), 4, m5=1.8)  # heap reuse
        one.free()
        many.free()
        other.close()
        after = free_bytes()
    assert before - after < 4 << 20  # 82 MB were allocated
