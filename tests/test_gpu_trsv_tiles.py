"""Triangular solves by tiles at the shapes where a tile can go wrong: ragged
boxes, grids with one line, entries that wrap round a grid line, rows of more
entries than a step holds in registers, rows beyond a tile's entries (a tile of
their own), more than 64 rows in a level, one row; every solve repeated (the solution arrays
alternate) and equal to the oracle bit for bit."""
import numpy as np
import pytest

import psblas3_amd as P
from test_gpu_spsv import _bits, _tri_mat, _vec

pytestmark = pytest.mark.gpu


def _csr(n, rows, rng, lower):
    """Triangle with the given strictly-lower column lists (mirrored for an upper
    one), the diagonal included, diagonally dominant."""
    irp, ja, val = [1], [], []
    for i in range(n):
        t = i if lower else n - 1 - i
        c = sorted(set(rows(t)))
        c = c if lower else [n - 1 - q for q in reversed(c)]
        v = list(rng.uniform(-1.0, 1.0, len(c)) / max(1, len(c)))
        c, v = (c + [i], v + [2.0]) if lower else ([i] + c, [2.0] + v)
        ja += [q + 1 for q in c]
        val += v
        irp.append(len(ja) + 1)
    return np.array(irp, np.int32), np.array(ja, np.int32), np.array(val)


def _grid(nx, ny, nz, wrap=False):
    def rows(t):
        x, y, z = t % nx, t // nx % ny, t // (nx * ny)
        c = [t - 1] if x > 0 or (wrap and t > 0) else []
        return c + ([t - nx] if y > 0 else []) + ([t - nx * ny] if z > 0 else [])
    return nx * ny * nz, rows


def _random(n, w, span, wide=0):
    rng = np.random.default_rng(n)
    cols = [rng.integers(max(0, t - span), t, wide if wide and t % 401 == 400 else w).tolist()
            if t else [] for t in range(n)]
    return n, lambda t: cols[t]


SHAPES = {"8x8x8": _grid(8, 8, 8), "9x8x17": _grid(9, 8, 17), "31x5x3": _grid(31, 5, 3),
          "2d_49x25": _grid(49, 25, 1), "2d_24x24": _grid(24, 24, 1),
          "wrap_16x9x4": _grid(16, 9, 4, wrap=True), "narrow_7x9x9": _grid(7, 9, 9),
          "chain_600": (600, lambda t: [t - 1] if t else []),
          "width4": _random(1500, 4, 40), "width6": _random(1500, 6, 600),
          "wide_rows": _random(2500, 3, 900, wide=300),
          "row_past_a_tile": _random(2500, 2, 2400, wide=1300),
          "levels_of_700": (4200, lambda t: [t - 700] if t >= 700 else []), "one": (1, lambda t: [])}


@pytest.mark.parametrize("name", list(SHAPES))
@pytest.mark.parametrize("lower,trans,single", [(True, "N", False), (False, "N", False),
                                                (True, "T", False), (False, "N", True)],
                         ids=["L", "U", "LT", "U-f32"])
def test_tiles_bitexact(gpu, orc, name, lower, trans, single):
    print(f"[gpu] case trsv tiles {name} lower={lower} trans={trans} single={single}", flush=True)
    n, rows = SHAPES[name]
    dt = np.float32 if single else np.float64
    irp, ja, val = _csr(n, rows, np.random.default_rng(5), lower)
    a, desc = _tri_mat(irp, ja, val, lower, False, single=single)
    for k in range(3):
        x = orc.uniform_pm1(30 + k, n).astype(dt)
        y0 = orc.uniform_pm1(40 + k, n).astype(dt)
        alpha, beta = [(1.0, 0.0), (2.0, -0.5), (-1.0, 0.0)][k]
        y = _vec(y0.copy(), single)
        P.psb_spsm(alpha, a, _vec(x, single), beta, y, desc, trans=trans)
        ref = orc.csr_cssv(irp, ja, val.astype(dt), x, lower=lower, trans=trans, alpha=alpha,
                           beta=beta, y=y0)
        assert np.array_equal(_bits(y.get_vect()), _bits(ref)), k
    a.free()


@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
def test_tiles_nonfinite(gpu, orc, single):
    """A right-hand side with infinities, NaN and the very pattern that marks an
    entry as not solved yet: the solve ends, and is non-finite where the
    oracle's is."""
    print(f"[gpu] case trsv tiles non-finite single={single}", flush=True)
    n, rows = _grid(11, 10, 9)
    dt = np.float32 if single else np.float64
    irp, ja, val = _csr(n, rows, np.random.default_rng(6), True)
    a, desc = _tri_mat(irp, ja, val, True, False, single=single)
    x = orc.uniform_pm1(50, n).astype(dt)
    x[n // 2] = np.inf
    x[n // 3] = np.nan
    unset = np.uint32(0x7FE5A3C9) if single else np.uint64(0x7FF8A5C3E1D2B497)
    x[n - 40] = np.array([unset]).view(dt)[0]
    y = _vec(np.zeros(n, dt), single)
    for _ in range(2):
        P.psb_spsm(1.0, a, _vec(x, single), 0.0, y, desc)
        ref = orc.csr_cssv(irp, ja, val.astype(dt), x)
        out = y.get_vect()
        assert np.array_equal(np.isnan(out), np.isnan(ref))
        ok = ~np.isnan(ref)
        assert np.array_equal(_bits(out[ok]), _bits(ref[ok]))
    a.free()


@pytest.mark.parametrize("nx,ny,nz", [(9, 9, 9), (25, 24, 1), (17, 15, 9), (41, 41, 5)])
@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
def test_tiles_ragged_arrays(gpu, orc, nx, ny, nz, single):
    """Row counts that do not fill the last line of a solution array, the last
    tile reading rows beside its own: twenty solves in turn in both arrays."""
    print(f"[gpu] case trsv tiles ragged {nx}x{ny}x{nz} single={single}", flush=True)
    n, rows = _grid(nx, ny, nz)
    dt = np.float32 if single else np.float64
    assert n * np.dtype(dt).itemsize % 128 != 0
    for lower in (True, False):
        irp, ja, val = _csr(n, rows, np.random.default_rng(8), lower)
        a, desc = _tri_mat(irp, ja, val, lower, False, single=single)
        x = orc.uniform_pm1(60, n).astype(dt)
        ref = orc.csr_cssv(irp, ja, val.astype(dt), x, lower=lower)
        for k in range(20):
            y = _vec(np.zeros(n, dt), single)
            P.psb_spsm(1.0, a, _vec(x, single), 0.0, y, desc)
            assert np.array_equal(_bits(y.get_vect()), _bits(ref)), k
        a.free()


def _bordered(n, full):
    """A chain with rows of all or so many earlier entries: full = {row: count}."""
    rng = np.random.default_rng(11)
    cols = {t: sorted(rng.choice(t - 1, c - 1, replace=False).tolist()) + [t - 1]
            for t, c in full.items()}
    return n, lambda t: cols.get(t, [t - 1] if t else [])


# 1024 entries still share a tile; 1025 do not; whole and ragged chunks of 1024;
# two wide rows in a row, the first possible and the last row
BORDERED = _bordered(3000, {1025: 1025, 1026: 1026, 1500: 1024, 2100: 2100, 2500: 2048,
                            2700: 2049, 2999: 2999})


@pytest.mark.parametrize("lower,trans,single", [(True, "N", False), (False, "N", False),
                                                (True, "T", False), (False, "T", True),
                                                (False, "N", True)],
                         ids=["L", "U", "LT", "UT-f32", "U-f32"])
def test_wide_rows_bitexact(gpu, orc, lower, trans, single):
    """Rows of more entries than a tile stages do not send the triangle to a launch
    per level.  For op 'T' the wide rows are those of the transpose, whose
    triangle is given."""
    print(f"[gpu] case trsv wide rows lower={lower} trans={trans} single={single}", flush=True)
    n, rows = BORDERED
    dt = np.float32 if single else np.float64
    irp, ja, val = _csr(n, rows, np.random.default_rng(12), lower if trans == "N" else not lower)
    if trans != "N":   # the transpose, diagonal last (lower) or first (upper) as stored rows are
        i = np.repeat(np.arange(1, n + 1), np.diff(irp))
        o = np.lexsort((i, ja))
        irp, ja, val = (np.concatenate([[1], 1 + np.cumsum(np.bincount(ja, minlength=n + 1)[1:])])
                        .astype(np.int32), i[o].astype(np.int32), val[o])
    a, desc = _tri_mat(irp, ja, val, lower, False, single=single)
    for k in range(3):
        x = orc.uniform_pm1(70 + k, n).astype(dt)
        y0 = orc.uniform_pm1(80 + k, n).astype(dt)
        alpha, beta = [(1.0, 0.0), (2.0, -0.5), (-1.0, 0.0)][k]
        y = _vec(y0.copy(), single)
        P.psb_spsm(alpha, a, _vec(x, single), beta, y, desc, trans=trans)
        ref = orc.csr_cssv(irp, ja, val.astype(dt), x, lower=lower, trans=trans, alpha=alpha,
                           beta=beta, y=y0)
        assert np.array_equal(_bits(y.get_vect()), _bits(ref)), k
    levels, tiles = a.a.sv_levels()
    assert levels == n and tiles > 7
    # in place: x and y the same vector
    x = orc.uniform_pm1(90, n).astype(dt)
    y = _vec(x.copy(), single)
    P.psb_spsm(1.0, a, y, 0.0, y, desc, trans=trans)
    assert np.array_equal(_bits(y.get_vect()),
                          _bits(orc.csr_cssv(irp, ja, val.astype(dt), x, lower=lower, trans=trans)))
    a.free()


def test_wide_row_ilu(gpu, orc):
    """The preconditioner's factors with wide rows, both as tiles."""
    import ctypes as C

    from psblas3_amd import _native as N
    print("[gpu] case trsv wide rows ilu", flush=True)
    n, rows = BORDERED
    f = {}
    for lower in (True, False):
        irp, ja, val = _csr(n, rows, np.random.default_rng(13), lower)
        keep = ja != np.repeat(np.arange(1, n + 1), np.diff(irp))       # unit factors
        f[lower] = (irp - np.arange(n + 1, dtype=np.int32),
                    ja[keep].astype(np.int32), val[keep])
    d = orc.uniform_pm1(14, n) + 2.0
    h = C.c_void_p()
    (li, lj, lv), (ui, uj, uv) = f[True], f[False]
    N.call("psb_hip_ilu_alloc", C.byref(h), n, li.ctypes.data, lj.ctypes.data, lv.ctypes.data,
           ui.ctypes.data, uj.ctypes.data, uv.ctypes.data, d.ctypes.data)
    ls, us = C.c_int(), C.c_int()
    N.call("psb_hip_ilu_segments", h, C.byref(ls), C.byref(us))
    assert ls.value > 7 and us.value > 7
    x = orc.uniform_pm1(15, n)
    xv, yv = P.psb_d_hip_vect().bld(x), P.psb_d_hip_vect().bld(np.zeros(n))
    xv.sync()
    yv.sync()
    N.call("psb_hip_ilu_apply", h, 1.0, xv.dev, 0.0, yv.dev)
    yv.set_dev()
    t = orc.csr_cssv(li, lj, lv, x, lower=True, unit=True)
    ref = orc.csr_cssv(ui, uj, uv, t * d, lower=False, unit=True)
    assert np.array_equal(_bits(yv.get_vect()), _bits(ref))
    N.call("psb_hip_ilu_free", h)
