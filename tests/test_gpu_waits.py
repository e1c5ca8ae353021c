"""Kernels whose workgroups wait for one another's values: when a wait is given
up (forced by a bound of one poll) the kernel ends, the next call that brings a
result to the host fails instead of handing out NaN, and with the usual bound
the same objects work again."""
import numpy as np
import pytest

import psblas3_amd as P
from psblas3_amd import _native as N
from test_gpu_spsv import _bits, _tri_mat, _vec

pytestmark = pytest.mark.gpu


@pytest.fixture
def one_poll(gpu):
    """Call it to bound every wait by one poll until the test ends; call it with 0
    for the usual bounds."""
    yield lambda polls=1: N.fn("psb_hip_set_wait_polls")(polls)
    N.fn("psb_hip_set_wait_polls")(0)


def _fails(f):
    with pytest.raises(N.PsbError) as e:
        f()
    assert e.value.info == N.RUNTIME and "wait" in str(e.value)


def test_triangular_solve(gpu, orc, one_poll):
    """A chain of 6,000 rows: eleven of its twelve tiles wait for the one before."""
    print("[gpu] case waits triangular solve", flush=True)
    n = 6000
    i = np.arange(n)
    irp = np.concatenate([[1, 2], 2 * i[1:] + 2]).astype(np.int32)
    ja = np.concatenate([[1], np.stack([i[1:], i[1:] + 1], 1).ravel()]).astype(np.int32)
    val = np.where(np.arange(2 * n - 1) % 2 == 0, 2.0, 0.5)
    a, desc = _tri_mat(irp, ja, val, True, False)
    x = orc.uniform_pm1(1, n)
    ref = orc.csr_cssv(irp, ja, val, x)
    y = _vec(np.zeros(n))

    def solve():
        P.psb_spsm(1.0, a, _vec(x), 0.0, y, desc)

    for result in (y.get_vect, lambda: P.psb_genrm2(y), lambda: N.call("psb_hip_device_sync")):
        solve()
        assert np.array_equal(_bits(y.get_vect()), _bits(ref))
        one_poll()
        solve()
        one_poll(0)
        _fails(result)
        N.call("psb_hip_device_sync")      # said once
    a.free()
