"""Vector operations by 16-byte loads at the sizes where they can go wrong:
remainders of a vector and of a thread's share, one grid-stride turn more or
less, more columns than one batch of results, infinities and NaN; a reduction
leaves the library stream idle."""
import ctypes as C
import math

import numpy as np
import pytest

import psblas3_amd as P
from psblas3_amd import _native as N

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def _vec(a):
    return (P.psb_s_hip_vect() if a.dtype == np.float32 else P.psb_d_hip_vect()).bld(a)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 2047, 2049, 65536, 65537, 1024 * 2048 - 1,
                               1024 * 2048 + 3, 3 * 1024 * 2048 + 1])
@pytest.mark.parametrize("dt", [np.float64, np.float32], ids=["f64", "f32"])
def test_sizes(gpu, orc, n, dt):
    print(f"[gpu] case vector ops n={n} {np.dtype(dt).name}", flush=True)
    x, y, z = (orc.uniform_pm1(100 + k, n).astype(dt) for k in range(3))
    xv, yv, zv = _vec(x), _vec(y), _vec(z)
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    # the products of FP64 entries round once, the sum in any order within
    # 2 log2(n) + 8 roundings (the blocks' trees and the 16 entries of a thread)
    bound = (2 * math.log2(max(n, 2)) + 8) * EPS
    assert abs(P.psb_gedot(xv, yv) - math.fsum(xd * yd)) <= bound * math.fsum(np.abs(xd * yd))
    assert abs(P.psb_genrm2(xv) ** 2 - math.fsum(xd * xd)) <= 2 * bound * math.fsum(xd * xd)
    assert abs(P.psb_geasum(xv) - math.fsum(np.abs(xd))) <= bound * math.fsum(np.abs(xd))
    assert P.psb_geamax(xv) == np.max(np.abs(xd))
    a, b = dt(0.7), dt(-0.3)
    P.psb_geaxpbyz(0.7, xv, -0.3, yv, zv)
    assert np.array_equal(zv.get_vect(), a * x + b * y)
    zv = _vec(z)
    P.psb_gemlt(0.7, xv, yv, -0.3, zv)
    assert np.array_equal(zv.get_vect(), b * z + a * y * x)


@pytest.mark.parametrize("cols", [1, 3, 33, 65])
def test_columns(gpu, orc, cols):
    """Every column's reduction, in batches of 32."""
    print(f"[gpu] case vector reductions cols={cols}", flush=True)
    n = 1001
    a = np.stack([orc.uniform_pm1(200 + c, n) for c in range(cols)], axis=1)
    v = _vec(a if cols > 1 else a[:, 0])
    got = np.atleast_1d(P.psb_genrm2(v))
    amax = np.atleast_1d(P.psb_geamax(v))
    for c in range(cols):
        one = _vec(a[:, c].copy())
        assert got[c] == P.psb_genrm2(one) and amax[c] == P.psb_geamax(one)


def test_nonfinite_and_empty(gpu):
    """Infinities and NaN come out as such; the scaled norm of huge entries;
    no entries give 0 (the results arrive, whatever they are)."""
    print("[gpu] case vector reductions non-finite", flush=True)
    x = np.ones(5000)
    x[1234] = np.inf
    xv, ones = _vec(x), _vec(np.ones(5000))
    assert P.psb_gedot(xv, ones) == np.inf and P.psb_geamax(xv) == np.inf
    x[77] = np.nan
    assert math.isnan(P.psb_gedot(_vec(x), ones))
    x[:] = np.array([np.uint64(0x7FF8D1E5A2C4B693)]).view(np.float64)[0]   # the waiting mark
    assert math.isnan(P.psb_gedot(_vec(x), ones))
    assert abs(P.psb_genrm2(_vec(np.full(5000, 1e300))) / (1e300 * math.sqrt(5000.0)) - 1) < 1e-14
    res = (C.c_double * 1)(7.0)
    N.call("psb_hip_mv_dot", res, 0, xv.dev, ones.dev)
    assert res[0] == 0.0


@pytest.mark.parametrize("n,cols", [(1, 1), (1001, 33), (4000003, 1)])
def test_reductions_synchronise(gpu, orc, n, cols):
    """A call that returns a host scalar synchronises the library stream
    (include/psb_hip.h): nothing is left on it, for any of the reductions."""
    print(f"[gpu] case reductions synchronise n={n} cols={cols}", flush=True)
    hip = C.CDLL("libamdhip64.so")
    stream = C.c_void_p(N.fn("psb_hip_get_stream")())
    v = _vec(np.full((n, cols) if cols > 1 else n, 0.5))
    P.psb_geaxpby(1.0, v, 0.0, v)
    res = (C.c_double * cols)()
    for name in ("psb_hip_mv_dot", "psb_hip_mv_nrm2", "psb_hip_mv_amax", "psb_hip_mv_asum"):
        for _ in range(20):
            N.call(name, res, n, v.dev, *([v.dev] if name == "psb_hip_mv_dot" else []))
            assert hip.hipStreamQuery(stream) == 0, name
