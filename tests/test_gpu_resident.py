"""Fused CG and BiCGSTAB whose vectors stay in registers over one launch of many
iterations, at the sizes where the split of rows changes (one row; one block and
one row more; the largest of each block size and rows per thread, and one row
more): the iterates and residual histories equal the host-driven reference
sequence's to rounding, over more iterations than one launch holds, in both
storage formats and from the allocation-free entry point."""
import numpy as np
import pytest

import psblas3_amd as P

pytestmark = pytest.mark.gpu

MOLDS = {"HLG": P.psb_d_hip_hlg_sparse_mat, "HLG32": lambda: P.psb_d_hip_hlg_sparse_mat(32),
         "ELG": P.psb_d_hip_elg_sparse_mat}


def _system(n, mold, spd, wide):
    """Diagonally dominant: a tridiagonal part, entries that reach other blocks
    (a third of the matrix away; 9973 rows away in the largest, whose columns
    are to fit in 16 bits), and two rows of 5 + wide slots."""
    if n == 1:
        return P.matrix_from_coo(1, 1, np.array([1], np.int32), np.array([1], np.int32),
                                 np.array([2.0]), mold=mold)
    i = np.arange(n, dtype=np.int32)
    rows, cols, vals = [i], [i], [6.0 + 0.1 * (i % 7)]
    for o, w in ((1, 1.0), (max(2, n // 3 if n <= 524288 else 9973), 0.5)):
        if o < n:
            rows += [i[o:], i[:-o]]
            cols += [i[:-o], i[o:]]
            vals += [np.full(n - o, -w), np.full(n - o, -w if spd else -0.6 * w)]
    if n > 256:
        r = np.array([n - 1, n // 2 + 3], np.int32).repeat(wide)
        c = r - 7 * np.tile(np.arange(1, wide + 1, dtype=np.int32), 2)
        rows += [r, c]
        cols += [c, r]
        vals += [np.full(r.size, -0.1), np.full(r.size, -0.1)]
    ia, ja, v = (np.concatenate(a) for a in (rows, cols, vals))
    return P.matrix_from_coo(n, n, ia.astype(np.int32) + 1, ja.astype(np.int32) + 1, v, mold=mold)


# wide: rows of more slots than the registers hold where a thread has one row,
# of seven and of eight where it has several
@pytest.mark.parametrize("fmt,n,wide", [("HLG", 1, 0), ("HLG", 257, 4), ("ELG", 1000, 12),
                                        ("HLG", 65536, 12), ("HLG", 65537, 20),
                                        ("HLG32", 100001, 3), ("ELG", 262144, 4),
                                        ("HLG", 262145, 2), ("ELG", 300000, 3),
                                        ("HLG", 524288, 3), ("HLG", 524289, 2),
                                        ("ELG", 700001, 3), ("HLG", 1048576, 2),
                                        ("HLG", 1048577, 2)])
@pytest.mark.parametrize("method", ["CG", "BICGSTAB"])
def test_resident_follows_reference_sequence(gpu, orc, fmt, n, wide, method):
    print(f"[gpu] case resident {fmt} n={n} wide={wide} {method}", flush=True)
    a = _system(n, MOLDS[fmt](), method == "CG", wide)
    desc = P.psb_cdall(nl=n)
    for ptype in ("DIAG", "NONE"):
        prec = P.psb_dprec_type(ptype).build(a, desc)
        b = P.vect_from(orc.uniform_pm1(3, n))
        # a few iterations of a well-conditioned system: rounding differences
        # of the sums (1e-16 relative, times the condition number, about 4, a
        # step) stay far below 1e-12
        its = 7
        x1, x2 = P.psb_geall(desc), P.psb_geall(desc)
        it1, e1, h1 = P.psb_krylov(method, a, prec, b, x1, 1e-14, desc, itmax=its)
        it2, e2, h2 = P.psb_krylov_fused(method, a, prec, b, x2, 1e-14, desc, itmax=its,
                                         history=True)
        assert it1 == it2
        m = min(len(h1), len(h2))
        h1, h2 = np.array(h1[:m]), np.array(h2[:m])
        assert np.all(np.abs(h1 - h2) <= 1e-12 * np.maximum(h1, 1e-2))
        r1, r2 = x1.get_vect(), x2.get_vect()
        assert np.linalg.norm(r1 - r2) <= 1e-12 * np.linalg.norm(r1)
        # again, and without allocations: the same bits, the entries were set back
        x3 = P.psb_geall(desc)
        P.psb_krylov_fused(method, a, prec, b, x3, 1e-14, desc, itmax=its)
        assert np.array_equal(x3.get_vect(), r2)
        if n <= 524288:
            x4 = P.psb_geall(desc)
            P.psb_krylov_fused(method, a, prec, b, x4, 1e-14, desc, itmax=its, noalloc=True)
            assert np.array_equal(x4.get_vect(), r2)
        prec.free()
    a.free()


@pytest.mark.parametrize("n", [3000, 70000])
def test_resident_over_several_launches(gpu, orc, n):
    """A 1-D Laplacian with a small shift takes hundreds of iterations: the
    vectors go through memory between launches, and the solution solves."""
    print(f"[gpu] case resident launches n={n}", flush=True)
    i = np.arange(n, dtype=np.int32)
    ia = np.concatenate([i[1:], i, i[:-1]]) + 1
    ja = np.concatenate([i[:-1], i, i[1:]]) + 1
    val = np.concatenate([np.full(n - 1, -1.0), np.full(n, 2.0 + 1e-3), np.full(n - 1, -1.0)])
    a = P.matrix_from_coo(n, n, ia, ja, val, mold=P.psb_d_hip_hlg_sparse_mat(64))
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type("NONE").build(a, desc)
    bh = orc.uniform_pm1(4, n)
    x = P.psb_geall(desc)
    it, err, hist = P.psb_krylov_fused("CG", a, prec, P.vect_from(bh), x, 1e-10, desc,
                                       itmax=5000, history=True)
    assert err <= 1e-10 and it > 100
    xh = x.get_vect()
    res = bh - ((2.0 + 1e-3) * xh - np.concatenate([[0.0], xh[:-1]])
                - np.concatenate([xh[1:], [0.0]]))
    # the recurrence's residual drifts from the true one by rounding of x only:
    # |A| eps |x| <= 4 * 1.1e-16 * 1e3 |b| a step, over it steps below 1e-9
    assert np.linalg.norm(res) <= 1e-9 * np.linalg.norm(bh)
    a.free()
