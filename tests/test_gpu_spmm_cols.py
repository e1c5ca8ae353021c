"""The multi-vector HLL product of narrow rows, column by column: each column
equals the single-vector product bit for bit, over hack widths around the
kernel's (5, 7, 9 slots), odd row counts, empty hacks, scattered columns (no
16-bit offsets) and hack sizes that leave one row per lane."""
import numpy as np
import pytest

import psblas3_amd as P

pytestmark = pytest.mark.gpu


def _matrix(kind, n, w, rng):
    i = np.arange(n)
    if kind == "band":        # up to w entries around the diagonal, a tenth left out
        off = [((k + 1) // 2) * (1 if k % 2 else -1) * (1 if k < 3 else 37) for k in range(w)]
        ia = np.concatenate([i for _ in off])
        ja = np.concatenate([i + o for o in off])
        ok = (ja >= 0) & (ja < n) & (rng.random(len(ja)) < 0.9)
        ia, ja = ia[ok], ja[ok]
    else:                     # w scattered columns; rows 64..127 empty
        ia = np.repeat(i[(i < 64) | (i >= 128)], w)
        ja = rng.integers(0, n, len(ia))
    return ia.astype(np.int32) + 1, ja.astype(np.int32) + 1, rng.uniform(-1.0, 1.0, len(ia))


@pytest.mark.parametrize("kind,n", [("band", 1), ("band", 1025), ("band", 4099),
                                    ("scattered", 70001)])
@pytest.mark.parametrize("w", [1, 5, 6, 7, 8, 9, 10])
@pytest.mark.parametrize("single,hk", [(False, 64), (False, 7), (True, 32)],
                         ids=["f64", "f64-hk7", "f32-hk32"])
def test_columns_bitexact(gpu, orc, kind, n, w, single, hk):
    print(f"[gpu] case spmm columns {kind} n={n} w={w} single={single} hk={hk}", flush=True)
    rng = np.random.default_rng(100 * w + n)
    ia, ja, val = _matrix(kind, n, w, rng)
    if not len(ia):
        ia, ja, val = np.array([1], np.int32), np.array([1], np.int32), np.array([2.0])
    mold = (P.psb_s_hip_hlg_sparse_mat if single else P.psb_d_hip_hlg_sparse_mat)(hk)
    vm = P.psb_s_hip_vect() if single else P.psb_d_hip_vect()
    dt = np.float32 if single else np.float64
    a = P.matrix_from_coo(n, n, ia, ja, val, mold=mold)
    for k, alpha, beta in ((2, 1.0, 0.0), (5, 2.0, -0.5)):
        X = np.stack([orc.uniform_pm1(70 + c, n) for c in range(k)], axis=1).astype(dt)
        Y0 = np.stack([orc.uniform_pm1(90 + c, n) for c in range(k)], axis=1).astype(dt)
        yv = vm.mold().bld(Y0)
        P.psb_spmm(alpha, a, vm.mold().bld(X), beta, yv)
        out = yv.get_vect()
        for c in range(k):
            y1 = vm.mold().bld(Y0[:, c].copy())
            P.psb_spmm(alpha, a, vm.mold().bld(X[:, c].copy()), beta, y1)
            assert np.array_equal(out[:, c], y1.get_vect()), (k, c)
    a.free()


@pytest.mark.parametrize("n,k,single", [
    (420000, 2, False), (420001, 2, False), (300000, 3, False), (300001, 4, False),
    (300000, 3, True), (300001, 3, True), (420001, 2, True), (2000, 4, True),
    (65536, 17, False), (65537, 17, False), (102400, 21, True), (102401, 21, True),
    (131072, 32, True), (131073, 32, True), (131072, 33, True)])
def test_either_side_of_the_lines(gpu, orc, n, k, single):
    """Row and column counts on both sides of the lines between columns one by one
    and in groups: first, last and a middle column equal the single-vector
    product bit for bit."""
    print(f"[gpu] case spmm lines n={n} k={k} single={single}", flush=True)
    ia, ja, val = _matrix("band", n, 7, np.random.default_rng(3))
    dt = np.float32 if single else np.float64
    vm = P.psb_s_hip_vect() if single else P.psb_d_hip_vect()
    a = P.matrix_from_coo(n, n, ia, ja, val,
                          mold=(P.psb_s_hip_hlg_sparse_mat if single
                                else P.psb_d_hip_hlg_sparse_mat)(64))
    X = np.stack([orc.uniform_pm1(70 + c, n) for c in range(k)], axis=1).astype(dt)
    yv = vm.mold().bld(np.zeros((n, k), dt))
    P.psb_spmm(1.5, a, vm.mold().bld(X), 0.0, yv)
    out = yv.get_vect()
    for c in {0, k // 2, k - 1}:
        y1 = vm.mold().bld(np.zeros(n, dt))
        P.psb_spmm(1.5, a, vm.mold().bld(X[:, c].copy()), 0.0, y1)
        assert np.array_equal(out[:, c], y1.get_vect()), c
    a.free()
