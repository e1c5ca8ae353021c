"""Kernels whose workgroups wait for one another's values: when a wait is given
up (forced from the host: no polls at all) the kernel ends, the next call that brings a
result to the host fails instead of handing out NaN, and with the usual bound
the same objects work again."""
import numpy as np
import pytest

import psblas3_amd as P
from psblas3_amd import _native as N
from test_gpu_spsv import _bits, _tri_mat, _vec

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_polls(gpu):
    """Call it to have every wait given up until the test ends; call it with 0 for
    the usual bounds."""
    yield lambda polls=-1: N.fn("psb_hip_set_wait_polls")(polls)
    N.fn("psb_hip_set_wait_polls")(0)


def _fails(f):
    with pytest.raises(N.PsbError) as e:
        f()
    assert e.value.info == N.RUNTIME and "wait" in str(e.value)


def test_triangular_solve(gpu, orc, no_polls):
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
        no_polls()
        solve()
        no_polls(0)
        _fails(result)
        N.call("psb_hip_device_sync")      # said once
    a.free()


def _poisson(L, mold):
    n = L ** 3
    g = np.arange(n, dtype=np.int32).reshape(L, L, L)
    ia, ja, val = [g.ravel()], [g.ravel()], [np.full(n, 6.0)]
    for ax in range(3):
        lo, hi = np.moveaxis(g, ax, 0)[:-1].ravel(), np.moveaxis(g, ax, 0)[1:].ravel()
        ia += [lo, hi]
        ja += [hi, lo]
        val += [np.full(2 * lo.size, -1.0)]
    return P.matrix_from_coo(n, n, np.concatenate(ia) + 1, np.concatenate(ja) + 1,
                             np.concatenate(val), mold=mold)


# iterations of one launch (HLG) and finalisations folded into launches per
# step (CSR, and rows beyond what the chip holds)
@pytest.mark.parametrize("fmt,L", [("HLG", 30), ("HLG", 64), ("CSRG", 64), ("HLG", 110)])
@pytest.mark.parametrize("method", ["CG", "BICGSTAB"])
def test_fused_solve(gpu, orc, no_polls, fmt, L, method):
    print(f"[gpu] case waits fused {fmt} L={L} {method}", flush=True)
    mold = P.psb_d_hip_hlg_sparse_mat(64) if fmt == "HLG" else P.psb_d_hip_csrg_sparse_mat()
    a = _poisson(L, mold)
    n = L ** 3
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type("DIAG").build(a, desc)
    b = P.vect_from(orc.uniform_pm1(2, n))
    noalloc = n * 8 * 10 < 64 << 20

    def solve(**kw):
        x = P.psb_geall(desc)
        it, err, _ = P.psb_krylov_fused(method, a, prec, b, x, 1e-8, desc, itmax=400, **kw)
        assert err <= 1e-8
        return it, x.get_vect()

    it, x = solve()
    no_polls()
    _fails(solve)
    if noalloc:
        _fails(lambda: solve(noalloc=True))
    no_polls(0)
    again = [solve()] + ([solve(noalloc=True)] if noalloc else [])
    assert all(i == it and np.array_equal(_bits(y), _bits(x)) for i, y in again)
    a.free()


@pytest.mark.parametrize("variant", ["restart", "reliable"])
def test_mixed_solve(gpu, orc, no_polls, variant):
    print(f"[gpu] case waits mixed {variant}", flush=True)
    a = _poisson(40, P.psb_d_hip_hlg_sparse_mat(64))
    n = 40 ** 3
    desc = P.psb_cdall(nl=n)
    prec = P.psb_dprec_type("DIAG").build(a, desc)
    b = P.vect_from(orc.uniform_pm1(3, n))

    def solve():
        x = P.psb_geall(desc)
        out = P.psb_krylov_mixed("CG", a, prec, b, x, 1e-10, desc, variant=variant)
        return out, x.get_vect()

    _, x = solve()
    no_polls()
    _fails(solve)
    no_polls(0)
    assert np.array_equal(_bits(solve()[1]), _bits(x))
    a.free()


@pytest.mark.parametrize("method,refine", [("CG", "reliable"), ("BICGSTAB", "restart"),
                                           ("BICGSTAB", "reliable")])
@pytest.mark.parametrize("graph", [True, False])
def test_batch_engine(gpu, orc, no_polls, method, refine, graph):
    """An engine one of whose waits was given up stays failed; another one works."""
    print(f"[gpu] case waits batch {method} {refine} graph={graph}", flush=True)
    coo = orc.gen_aniso2d(70, 0.5)        # 5 tiles
    a = P.matrix_from_coo(coo.nr, coo.nc, coo.ia, coo.ja, coo.val,
                          mold=P.psb_d_hip_hlg_sparse_mat(64))
    prec = P.psb_dprec_type("DIAG").build(a, P.psb_cdall(nl=coo.nr))
    b = P.vect_from(orc.uniform_pm1(4, coo.nr))

    def engine():
        eng = P.psb_hip_batch(method, max_systems=4, arena_bytes=16 << 20, refine=refine,
                              use_graph=graph)
        return eng, eng.register(a, prec)

    no_polls()
    eng, mid = engine()
    _fails(lambda: eng.solve([(mid, b, P.psb_d_hip_vect().all(coo.nr))], eps=1e-6, itmax=500))
    no_polls(0)
    _fails(eng.step)
    _fails(eng.poll)
    eng.free()
    N.call("psb_hip_device_sync")          # the engine's failure is its own
    eng, mid = engine()
    res = eng.solve([(mid, b, P.psb_d_hip_vect().all(coo.nr))], eps=1e-6, itmax=500)
    assert res[0]["status"] == 1
    eng.free()
