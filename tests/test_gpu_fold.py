"""Fused CG and BiCGSTAB whose kernels apply their own finalisation, at the grid
sizes where that can go wrong (one block, a ragged last block, the largest
folded grid and one block more, where a launch of its own finalises): the
iterates and residual histories of a few iterations equal the host-driven
reference sequence's to rounding."""
import numpy as np
import pytest

import psblas3_amd as P

pytestmark = pytest.mark.gpu


def _system(n, mold, spd):
    """Tridiagonal, diagonally dominant, with a far coupling."""
    i = np.arange(n, dtype=np.int32)
    far = max(2, n // 3)
    ia = np.concatenate([i[1:], i, i[:-1], i[far:], i[:-far]]) + 1
    ja = np.concatenate([i[:-1], i, i[1:], i[:-far], i[far:]]) + 1
    up = -1.0 if spd else -0.6
    val = np.concatenate([np.full(n - 1, -1.0), 5.0 + 0.1 * (i % 7), np.full(n - 1, up),
                          np.full(n - far, -0.5), np.full(n - far, -0.5)]) if n > far else \
        np.full(len(ia), 5.0)
    return P.matrix_from_coo(n, n, ia, ja, val, mold=mold)


FOLD = 8192 * 512     # rows of the largest folded FP64 product
MOLDS = {"HLG": P.psb_d_hip_hlg_sparse_mat, "ELG": P.psb_d_hip_elg_sparse_mat,
         "CSRG": P.psb_d_hip_csrg_sparse_mat}


@pytest.mark.parametrize("fmt,n", [("HLG", 1), ("HLG", 300), ("HLG", 513), ("ELG", 100001),
                                   ("CSRG", 100001), ("HLG", FOLD), ("HLG", FOLD + 1)])
@pytest.mark.parametrize("method", ["CG", "BICGSTAB"])
def test_fused_follows_reference_sequence(gpu, orc, fmt, n, method):
    print(f"[gpu] case fold {fmt} n={n} {method}", flush=True)
    if n == 1:
        a = P.matrix_from_coo(1, 1, np.array([1], np.int32), np.array([1], np.int32),
                              np.array([2.0]), mold=MOLDS[fmt]())
    else:
        a = _system(n, MOLDS[fmt](), method == "CG")
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type("DIAG").build(a, desc)
    b = P.vect_from(orc.uniform_pm1(3, n))
    its = 6
    # 6 iterations of a well-conditioned system: rounding differences of the
    # sums (1e-16 relative, times the condition number, about 3, a step) stay
    # far below 1e-12
    x1, x2 = P.psb_geall(desc), P.psb_geall(desc)
    it1, e1, h1 = P.psb_krylov(method, a, prec, b, x1, 1e-14, desc, itmax=its)
    it2, e2, h2 = P.psb_krylov_fused(method, a, prec, b, x2, 1e-14, desc, itmax=its, history=True)
    assert it1 == it2
    m = min(len(h1), len(h2))
    h1, h2 = np.array(h1[:m]), np.array(h2[:m])
    assert np.all(np.abs(h1 - h2) <= 1e-12 * np.maximum(h1, 1e-2))
    r1, r2 = x1.get_vect(), x2.get_vect()
    assert np.linalg.norm(r1 - r2) <= 1e-12 * np.linalg.norm(r1)
    # twice the same solve: the slots were set back
    x3 = P.psb_geall(desc)
    P.psb_krylov_fused(method, a, prec, b, x3, 1e-14, desc, itmax=its)
    assert np.array_equal(x3.get_vect(), r2)
    a.free()
