"""Fused CG and BiCGSTAB whose vectors stay in registers over one launch of many
iterations, at the sizes where the split of rows changes (one row; one block and
one row more; the largest of each block size and rows per thread, and one row
more): the iterates and residual histories equal the host-driven reference
sequence's to rounding, in both storage formats and from the allocation-free
entry point; over several launches, in both precisions; and where a launch
finds the chip taken and the solve goes on with launches per step."""
import numpy as np
import pytest

import psblas3_amd as P
from psblas3_amd import _native as N

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


# wide: rows of more slots than the registers hold where a thread has one row
# (over 8), of seven and of eight where it has several, and of more than those
# hold there, which take launches per step
@pytest.mark.parametrize("fmt,n,wide", [("HLG", 1, 0), ("HLG", 257, 4), ("ELG", 1000, 12),
                                        ("HLG", 65536, 12), ("HLG", 65537, 20),
                                        ("HLG32", 100001, 3), ("ELG", 262144, 4),
                                        ("HLG", 262145, 2), ("ELG", 300000, 3),
                                        ("HLG", 300001, 6), ("ELG", 700001, 5),
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


@pytest.fixture
def leave(gpu):
    """leave(k): every solve leaves at its k-th resident launch (0: none) until the
    test ends; returns how many have left since the call before."""
    f = N.fn("psb_hip_set_resident_leave")
    f(0)
    yield f
    f(0)


def _chain(n, method, mold, single=False):
    """A chain whose solve takes over 130 iterations and whose residuals two ways
    of adding the sums leave alike (_alike).  For CG a shift of 1e-3, no Ritz
    value converges, and entries 9,973 rows away reach other blocks; for
    BiCGSTAB a skew chain with a shift of 0.1."""
    i = np.arange(n, dtype=np.int32)
    if method == "CG":
        lo, up, dg = -1.0, -1.0, 2.003
    else:
        lo, up, dg = -1.3, -0.7, 2.1
    rows, cols = [i[1:], i, i[:-1]], [i[:-1], i, i[1:]]
    vals = [np.full(n - 1, lo), np.full(n, dg), np.full(n - 1, up)]
    o = 9973
    if method == "CG" and n > o:
        rows += [i[o:], i[:-o]]
        cols += [i[:-o], i[o:]]
        vals += [np.full(n - o, -1e-3), np.full(n - o, -1e-3)]
    val = np.concatenate(vals).astype(np.float32 if single else np.float64)
    return P.matrix_from_coo(n, n, np.concatenate(rows) + 1, np.concatenate(cols) + 1, val,
                             mold=mold)


def _resident(leave, solve):
    """Whether the solve is a resident one."""
    leave(1)
    solve()
    return leave(0) == 1


S_HLG = P.psb_s_hip_hlg_sparse_mat


def _histories(orc, fmt, n, method, ptype, its, single=False):
    mold = S_HLG(64) if single else (P.psb_d_hip_hlg_sparse_mat(64) if fmt == "HLG"
                                     else MOLDS[fmt]())
    a = _chain(n, method, mold, single)
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type(ptype).build(a, desc)

    def vect(v):
        return P.vect_from(v.astype(np.float32), mold=P.psb_s_hip_vect()) if single \
            else P.vect_from(v)
    b = vect(orc.uniform_pm1(3, n))

    def run(solver, **kw):
        x = vect(np.zeros(n))
        it, _, h = solver(method, a, prec, b, x, 1e-30, desc, itmax=its, **kw)
        return it, np.array(h), x.get_vect()
    return run


def _alike(method, its, one, other):
    """Histories and iterates of two solves of a _chain.  The same recurrences in
    numpy with two orders of summation differ, over 130 iterations, three sizes
    and six right-hand sides, for CG by 4.2e-15 at most, for BiCGSTAB by 5e-6 on
    nine iterations of ten and up to 2e-3 where a denominator comes near zero; a
    vector lost on the way makes nearly all that follow differ by their size."""
    (it1, h1, x1), (it2, h2, x2) = one, other
    assert it1 == it2 == its and min(len(h1), len(h2)) >= its - 1
    m = min(len(h1), len(h2))
    d = np.abs(h1[:m] - h2[:m]) / h1[:m]
    assert d.max() <= 1e-12 if method == "CG" else np.quantile(d, 0.9) <= 1e-3
    assert np.linalg.norm(x1 - x2) <= 1e-12 * np.linalg.norm(x1)


CHAINS = [("HLG", 3000, "CG", "DIAG"), ("HLG", 3001, "CG", "NONE"), ("ELG", 100000, "CG", "DIAG"),
          ("HLG", 400001, "CG", "DIAG"), ("ELG", 500000, "CG", "NONE"),
          ("HLG", 700001, "CG", "DIAG"), ("ELG", 1000000, "CG", "DIAG"),
          ("HLG", 3000, "BICGSTAB", "DIAG"), ("ELG", 200001, "BICGSTAB", "DIAG"),
          ("ELG", 400001, "BICGSTAB", "DIAG"), ("HLG", 500000, "BICGSTAB", "NONE")]


@pytest.mark.parametrize("fmt,n,method,ptype", CHAINS)
def test_state_through_launches(gpu, orc, leave, fmt, n, method, ptype):
    """110 iterations, three launches of 48: residual history and iterate follow the
    reference sequence's, one, two and four rows a thread, p, z, r and v through
    memory between launches."""
    print(f"[gpu] case resident state {fmt} n={n} {method} {ptype}", flush=True)
    its = 110
    run = _histories(orc, fmt, n, method, ptype, its)
    assert _resident(leave, lambda: run(P.psb_krylov_fused, history=True))
    _alike(method, its, run(P.psb_krylov), run(P.psb_krylov_fused, history=True))


@pytest.mark.parametrize("n", [3000, 100001, 400001, 900001])
def test_state_through_launches_fp32(gpu, orc, leave, n):
    """The same in single precision (CG), against launches per step: the vectors
    take the same roundings, only the FP64 sums another order, so alpha and beta
    differ by a unit in the last FP32 place now and then (6e-8)."""
    print(f"[gpu] case resident state fp32 n={n}", flush=True)
    its = 110
    run = _histories(orc, "HLG", n, "CG", "DIAG", its, single=True)
    leave(1)
    it1, h1, x1 = run(P.psb_krylov_fused, history=True)
    assert leave(0) == 1
    it2, h2, x2 = run(P.psb_krylov_fused, history=True)
    assert leave(0) == 0 and it1 == it2 == its
    # a unit in the last place in each of 110 steps would be 110 * 6e-8
    assert np.all(np.abs(h1 - h2) <= 1e-5 * h1)
    assert np.linalg.norm(x1 - x2) <= 1e-5 * np.linalg.norm(x1)


@pytest.mark.parametrize("at", [1, 2, 3])
@pytest.mark.parametrize("fmt,n,method,ptype", [CHAINS[0], CHAINS[1], CHAINS[3], CHAINS[6],
                                                CHAINS[7], CHAINS[8], CHAINS[10]])
def test_chip_taken_mid_solve(gpu, orc, leave, fmt, n, method, ptype, at):
    """The launch finds the chip taken: the solve goes on from there with launches
    per step, the same recurrence from the entry points with and without
    allocations."""
    print(f"[gpu] case resident leave {fmt} n={n} {method} {ptype} at={at}", flush=True)
    its = 130
    run = _histories(orc, fmt, n, method, ptype, its)
    ref = run(P.psb_krylov)
    for kw in ({}, {"noalloc": True}):
        leave(at)
        got = run(P.psb_krylov_fused, history=True, **kw)
        assert leave(0) == 1
        _alike(method, its, ref, got)


@pytest.mark.parametrize("at", [1, 2, 3])
@pytest.mark.parametrize("variant", ["restart", "reliable"])
@pytest.mark.parametrize("ptype,n", [("DIAG", 100001), ("NONE", 100001), ("DIAG", 400001),
                                     ("DIAG", 900001)])
def test_chip_taken_mixed(gpu, orc, leave, variant, ptype, n, at):
    """Mixed precision, one, two and four rows a thread: the inner solve's launch finds
    the chip taken; the solution
    and the number of inner iterations are those of the undisturbed solve to the
    roundings of the sums."""
    print(f"[gpu] case resident leave mixed {variant} {ptype} n={n} at={at}", flush=True)
    a = _chain(n, "CG", P.psb_d_hip_hlg_sparse_mat(64))
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type(ptype).build(a, desc)
    b = P.vect_from(orc.uniform_pm1(5, n))
    out = []
    for k in (0, at):
        leave(k)
        x = P.psb_geall(desc)
        outer, inner, err = P.psb_krylov_mixed("CG", a, prec, b, x, 1e-10, desc,
                                               variant=variant)
        assert err <= 1e-10
        out.append((inner, x.get_vect()))
    assert leave(0) == 1
    (i0, x0), (i1, x1) = out
    # two solutions of residual 1e-10 |b| differ by at most 2e-10 |b| / 1e-3, the
    # smallest eigenvalue; |x| is at least |b| / 4.1
    assert np.linalg.norm(x0 - x1) <= 1e-6 * np.linalg.norm(x0)
    # a lost direction would cost about another half solve; roundings a few steps
    assert abs(i0 - i1) <= 4 + i0 // 20
    a.free()


def test_taken_chip_is_remembered(gpu, orc, leave):
    """After a solve that left, the solves of the next second do not try."""
    print("[gpu] case resident leave remembered", flush=True)
    run = _histories(orc, "HLG", 3000, "CG", "DIAG", 60)
    leave(1)
    got = [run(P.psb_krylov_fused) for _ in range(4)]
    assert leave(1) == 1
    assert all(np.array_equal(got[0][2], g[2]) for g in got)
    run(P.psb_krylov_fused)
    assert leave(0) == 1


@pytest.mark.parametrize("method,n,wide,resident", [
    ("CG", 1048576, 2, True), ("CG", 1048577, 2, False), ("BICGSTAB", 524288, 3, True),
    ("BICGSTAB", 524289, 2, False), ("CG", 300001, 3, True), ("CG", 300001, 6, False),
    ("CG", 65537, 39, True), ("CG", 65537, 40, False), ("CG", 65536, 43, True),
    ("CG", 65536, 44, False), ("CG", 8192, 145, True), ("CG", 8192, 146, False),
    ("CG", 8193, 99, True), ("CG", 8193, 100, False), ("CG", 131073, 83, True),
    ("CG", 131073, 84, False)])
def test_which_solves_are_resident(gpu, orc, leave, method, n, wide, resident):
    """More rows than the threads hold, several a thread wider than eight slots, or
    rows too wide to gain by it (5 + wide slots), take launches per step."""
    print(f"[gpu] case resident rule {method} n={n} wide={wide}", flush=True)
    a = _system(n, P.psb_d_hip_hlg_sparse_mat(64), method == "CG", wide)
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type("DIAG").build(a, desc)
    b = P.vect_from(orc.uniform_pm1(3, n))
    assert resident == _resident(leave, lambda: P.psb_krylov_fused(
        method, a, prec, b, P.psb_geall(desc), 1e-14, desc, itmax=3))
    a.free()
