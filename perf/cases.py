"""The work a program that uses this package has the GPU do: sparse products in
every storage format, multi-vector products, triangular solves, the vector
operations of a Krylov loop, whole Krylov solves and a batch of them.

Every matrix is made here, from the seed: 7-point convection-diffusion and
Poisson stencils on an L^3 grid and 5-point anisotropic ones on an L^2 grid
(assembled with psb_spall / psb_spins / psb_spasb, as a PDE code does), and
matrices of power-law rows with scattered columns (graphs).
"""
import math

import numpy as np
import torch

import psblas3_amd as P
from psblas3_amd import _native as N

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one product of a small grid problem: launch and call latency count
        {"name": "spmv_hll_f64_L40", "kind": "spmv", "fmt": "HLG", "dtype": "d", "L": 40,
         "trans": "N"},
        # the product of a large grid problem, matrix and vectors past the caches
        {"name": "spmv_hll_f64_L200", "kind": "spmv", "fmt": "HLG", "dtype": "d", "L": 200,
         "trans": "N"},
        # single precision, ELL storage, an odd grid (ragged last tile)
        {"name": "spmv_ell_f32_L161", "kind": "spmv", "fmt": "ELG", "dtype": "s", "L": 161,
         "trans": "N"},
        # the CSR storage a program keeps when it also solves with the matrix
        {"name": "spmv_csr_f64_L137", "kind": "spmv", "fmt": "CSRG", "dtype": "d", "L": 137,
         "trans": "N"},
        # rows of very uneven length with scattered columns (a graph)
        {"name": "spmv_csr_f64_graph_2M", "kind": "graph", "fmt": "CSRG", "dtype": "d",
         "n": 2000000},
        # several right-hand sides at once: block methods, multiple loads
        {"name": "spmm_hll_f64_L160_k8", "kind": "spmm", "dtype": "d", "L": 160, "k": 8},
        {"name": "spmm_hll_f64_L100_k32", "kind": "spmm", "dtype": "d", "L": 100, "k": 32},
        # a forward sweep with the lower triangle (Gauss-Seidel, psb_spsm)
        {"name": "spsm_csr_f64_L64", "kind": "spsm", "dtype": "d", "L": 64, "lower": True,
         "trans": "N"},
        # the vector steps of a Krylov iteration, from the smallest to streaming sizes
        {"name": "vector_f64_1M", "kind": "vector", "dtype": "d", "n": 1000003},
        # a whole solve through the reference's call sequence, ILU(0) preconditioned
        {"name": "krylov_bicgstab_bjac_L40", "kind": "krylov", "method": "BICGSTAB",
         "prec": "BJAC", "L": 40},
        # a whole solve with every scalar kept on the device
        {"name": "fused_cg_f64_L100", "kind": "fused", "method": "CG", "fmt": "HLG",
         "mixed": False, "L": 100},
        # many independent systems of uneven sizes advancing together
        {"name": "batch_cg_24", "kind": "batch", "nsys": 24, "lmin": 32, "lmax": 256},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "graph", "spmm", "spmm", "spsm", "vector",
                       "krylov", "fused", "batch"])
    dt = rng.choice(["d", "d", "s"])
    if kind == "spmv":
        return {"kind": kind, "fmt": rng.choice(["HLG", "ELG", "CSRG"]), "dtype": dt,
                "L": _logint(rng, 24, 180), "trans": rng.choice(["N", "N", "N", "T"])}
    if kind == "graph":
        return {"kind": kind, "fmt": rng.choice(["CSRG", "HLGS"]), "dtype": dt,
                "n": _logint(rng, 100000, 2000000)}
    if kind == "spmm":
        k = rng.choice([2, 3, 4, 6, 8, 12, 16, 24, 32])
        return {"kind": kind, "dtype": dt, "L": _logint(rng, 32, min(150, int((32e6 / k) ** (1 / 3)))),
                "k": k}
    if kind == "spsm":
        return {"kind": kind, "dtype": dt, "L": _logint(rng, 24, 110),
                "lower": rng.choice([True, False]), "trans": rng.choice(["N", "N", "T"])}
    if kind == "vector":
        return {"kind": kind, "dtype": dt, "n": _logint(rng, 20000, 8000000)}
    if kind == "krylov":
        method = rng.choice(["BICGSTAB", "CG", "RGMRES"])
        return {"kind": kind, "method": method,
                "prec": "BJAC" if method == "RGMRES" else rng.choice(["BJAC", "DIAG"]),
                "L": _logint(rng, 24, 60)}
    if kind == "fused":
        mixed = rng.choice([False, False, True])
        return {"kind": kind, "method": "CG" if mixed else rng.choice(["CG", "BICGSTAB"]),
                "fmt": "HLG" if mixed else rng.choice(["HLG", "ELG", "CSRG"]), "mixed": mixed,
                "L": _logint(rng, 24, 110)}
    return {"kind": "batch", "nsys": rng.randint(6, 24), "lmin": 32, "lmax": rng.randint(64, 256)}


# ------------------------------------------------------------------ inputs
def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * (seed + 1) + stream)
    return g


def _rand(seed, stream, *shape, single=False):
    """Uniform in [-1, 1), float64 (of single-precision values when single)."""
    u = 2.0 * torch.rand(*shape, generator=_gen(seed, stream), device=DEV,
                         dtype=torch.float64) - 1.0
    return u.float().double() if single else u


def _stencil(L, seed, spd=False, jitter=0.5, single=False):
    """7-point stencil on L^3: row r couples to r + off[k] with C[k, r] (0 outside the
    grid).  Convection of a seeded magnitude in [0, 10) (none when spd), the diagonal
    raised by up to jitter row by row."""
    n, h = L ** 3, 1.0 / (L + 1)
    conv = 0.0 if spd else 5.0 * float(_rand(seed, 7, 1).item() + 1.0)
    c = conv * h / (2.0 * math.sqrt(3.0))
    r = torch.arange(n, device=DEV)
    x, y, z = r % L, (r // L) % L, r // (L * L)
    off = [-L * L, -L, -1, 0, 1, L, L * L]
    inside = [z > 0, y > 0, x > 0, None, x < L - 1, y < L - 1, z < L - 1]
    C = torch.empty(7, n, device=DEV, dtype=torch.float64)
    for k in range(7):
        if k == 3:
            C[k] = 6.0 + (jitter * 0.5 * (_rand(seed, 8, n) + 1.0) if jitter else 0.0)
        else:
            C[k] = torch.where(inside[k], -1.0 - c if k < 3 else -1.0 + c, 0.0)
    return off, (C.float().double() if single else C)


def _aniso(L, e):
    """5-point -e u_xx - u_yy on L^2, as _stencil gives it."""
    n = L * L
    r = torch.arange(n, device=DEV)
    x, y = r % L, r // L
    C = torch.empty(5, n, device=DEV, dtype=torch.float64)
    C[0] = torch.where(y > 0, -1.0, 0.0)
    C[1] = torch.where(x > 0, -e, 0.0)
    C[2] = 2.0 + 2.0 * e
    C[3] = torch.where(x < L - 1, -e, 0.0)
    C[4] = torch.where(y < L - 1, -1.0, 0.0)
    return [-L, -1, 0, 1, L], C


def _apply(off, C, x):
    """A x (columns of x apart) in float64; with C's k-th row moved it is also A^T x."""
    n = C.shape[1]
    y = torch.zeros_like(x)
    for o, c in zip(off, C):
        lo, hi = max(0, -o), min(n, n - o)
        cc = c[lo:hi] if x.ndim == 1 else c[lo:hi, None]
        y[lo:hi] += cc * x[lo + o:hi + o]
    return y


def _transposed(off, C):
    """A^T in the same form."""
    T = torch.zeros_like(C)
    n = C.shape[1]
    for k, o in enumerate(off):   # A[r, r+o] = C[k, r]  ->  A^T[r+o, r], offset -o
        lo, hi = max(0, -o), min(n, n - o)
        T[len(off) - 1 - k, lo + o:hi + o] = C[k, lo:hi]
    return [-o for o in reversed(off)], T


def _triplets(off, C):
    n = C.shape[1]
    keep = (C != 0.0).T
    r = torch.arange(n, device=DEV, dtype=torch.int32)
    o = torch.tensor(off, device=DEV, dtype=torch.int32)
    ia = (r[:, None] + 1).expand(n, len(off))[keep]
    ja = (r[:, None] + 1 + o[None, :])[keep]
    return n, ia.cpu().numpy(), ja.cpu().numpy(), C.T[keep].cpu().numpy()


def _graph(n, seed, single):
    """Rows of power-law length (mean about 16, at most 4096), columns uniform."""
    u = 0.5 * (_rand(seed, 20, n) + 1.0)
    ln = torch.clamp(5.4 * torch.pow(1.0 - u, -1.0 / 1.5), max=4096.0).to(torch.int64)
    ia = torch.repeat_interleave(torch.arange(n, device=DEV), ln)
    nnz = ia.numel()
    ja = torch.randint(0, n, (nnz,), generator=_gen(seed, 21), device=DEV)
    # multiples of 2^-10, so that a duplicate entry's sum is the same in either precision
    val = torch.randint(-1024, 1024, (nnz,), generator=_gen(seed, 22),
                        device=DEV).double() / 1024.0
    return ia, ja, val


def _vector_input(case, seed, j):
    """p, q, r of a vector case, and its inverse diagonal d (positive) for j = 3."""
    u = _rand(seed, j, case["n"], single=case["dtype"] == "s")
    return (0.5 + 0.25 * u).float().double() if j == 3 else u


_MOLD = {("HLG", "d"): lambda: P.psb_d_hip_hlg_sparse_mat(64),
         ("HLG", "s"): lambda: P.psb_s_hip_hlg_sparse_mat(64),
         ("HLGS", "d"): lambda: P.psb_d_hip_hlg_sparse_mat(64, sort_window=0),
         ("HLGS", "s"): lambda: P.psb_s_hip_hlg_sparse_mat(64, sort_window=0),
         ("ELG", "d"): lambda: P.psb_d_hip_elg_sparse_mat(),
         ("ELG", "s"): lambda: P.psb_s_hip_elg_sparse_mat(),
         ("CSRG", "d"): lambda: P.psb_d_hip_csrg_sparse_mat(),
         ("CSRG", "s"): lambda: P.psb_s_hip_csrg_sparse_mat()}


def _matrix(off, C, fmt, dt="d"):
    n, ia, ja, val = _triplets(off, C)
    return P.matrix_from_coo(n, n, ia, ja, val, mold=_MOLD[fmt, dt]())


class _Memory:
    """A device vector's memory as torch takes it."""

    def __init__(self, v):
        kind = "<f8" if v._dtype == np.float64 else "<f4"
        es = int(kind[2])
        pitch = N.fn("psb_hip_mv_pitch")(v.dev)
        self.owner = v
        self.__cuda_array_interface__ = {
            "shape": (v.n,) if v.count == 1 else (v.count, v.n), "typestr": kind, "version": 2,
            "strides": None if v.count == 1 else (pitch * es, es),
            "data": (int(N.fn("psb_hip_mv_data")(v.dev)), False)}


def _vector(n, dt="d", k=1, values=None):
    """(a device vector of n entries and k columns, its memory as a tensor)."""
    v = (P.psb_d_hip_vect() if dt == "d" else P.psb_s_hip_vect()).all(n, k)
    t = torch.as_tensor(_Memory(v), device=DEV)
    P.psb_hip_DeviceSync()
    if values is not None:
        t.copy_(values if k == 1 else values.T)
        torch.cuda.synchronize()
    v.set_dev()
    return P.psb_d_vect_type(v), t


def prepare(case, seed):
    P.psb_init(0)
    kind, dt = case["kind"], case.get("dtype", "d")
    single = dt == "s"
    s = {"case": case}
    if kind == "spmv":
        off, C = _stencil(case["L"], seed, single=single)
        s["a"] = _matrix(off, C, case["fmt"], dt)
        n = C.shape[1]
        s["x"], _ = _vector(n, dt, values=_rand(seed, 1, n, single=single))
        s["y"], s["ty"] = _vector(n, dt)
        if case["trans"] == "T":   # the transpose is built with the first product
            P.psb_spmm(1.0, s["a"], s["x"], 0.0, s["y"], trans="T")
    elif kind == "graph":
        n = case["n"]
        ia, ja, val = _graph(n, seed, single)
        s["a"] = P.matrix_from_coo(n, n, (ia + 1).int().cpu().numpy(),
                                   (ja + 1).int().cpu().numpy(), val.cpu().numpy(),
                                   mold=_MOLD[case["fmt"], dt]())
        s["x"], _ = _vector(n, dt, values=_rand(seed, 1, n, single=single))
        s["y"], s["ty"] = _vector(n, dt)
    elif kind == "spmm":
        off, C = _stencil(case["L"], seed, single=single)
        s["a"] = _matrix(off, C, "HLG", dt)
        n, k = C.shape[1], case["k"]
        s["x"], _ = _vector(n, dt, k, values=_rand(seed, 1, n, k, single=single))
        s["y"], s["ty"] = _vector(n, dt, k)
    elif kind == "spsm":
        off, C = _stencil(case["L"], seed, single=single)
        n = C.shape[1]
        C = C.clone()
        C[4:] = 0.0 if case["lower"] else C[4:]
        C[:3] = C[:3] if case["lower"] else 0.0
        s["a"] = _matrix(off, C, "CSRG", dt)
        s["a"].set_triangle()
        s["a"].set_lower(case["lower"])
        s["x"], _ = _vector(n, dt, values=_rand(seed, 1, n, single=single))
        s["y"], s["ty"] = _vector(n, dt)
        # the level analysis is made with the first solve and kept with the matrix
        P.psb_spsm(1.0, s["a"], s["x"], 0.0, s["y"], trans=case["trans"])
    elif kind == "vector":
        n = case["n"]
        for j, name in enumerate("pqrd"):
            s[name], _ = _vector(n, dt, values=_vector_input(case, seed, j))
        for name in "xyz":
            s[name], s["t" + name] = _vector(n, dt)
    elif kind == "krylov" or kind == "fused":
        spd = case["method"] == "CG"
        off, C = _stencil(case["L"], seed, spd=spd, jitter=0.0)
        n = C.shape[1]
        s["a"] = _matrix(off, C, case.get("fmt", "HLG"))
        s["desc"] = P.psb_cdall(nl=n)
        s["prec"] = P.psb_dprec_type(case.get("prec", "DIAG")).build(s["a"], s["desc"])
        s["b"], _ = _vector(n, values=_apply(off, C, _rand(seed, 1, n)))
        s["x"], s["tx"] = _vector(n)
    elif kind == "batch":
        systems, total = _systems(case, seed), 0
        s["mats"], s["jobs"], s["tx"] = [], [], []
        for off, C, xt in systems:
            n = C.shape[1]
            a = _matrix(off, C, "HLG")
            prec = P.psb_dprec_type("DIAG").build(a, P.psb_cdall(nl=n))
            b, _ = _vector(n, values=_apply(off, C, xt))
            x, tx = _vector(n)
            total += 3 * ((8 * n + 255) // 256 * 256) + 5 * ((4 * n + 255) // 256 * 256)
            s["mats"].append((a, prec))
            s["jobs"].append([None, b, x])
            s["tx"].append(tx)
        s["eng"] = P.psb_hip_batch("CG", max_systems=len(systems), arena_bytes=total + (1 << 20))
        for j, (a, prec) in zip(s["jobs"], s["mats"]):
            j[0] = s["eng"].register(a, prec)
    P.psb_hip_DeviceSync()
    return s


def _systems(case, seed):
    """Anisotropic 2-D problems, sides spread over [lmin, lmax] in their logarithm."""
    m, out = case["nsys"], []
    es = torch.pow(10.0, -1.5 + 1.5 * _rand(seed, 30, m)).tolist()
    for k in range(m):
        L = int(round(case["lmin"] * (case["lmax"] / case["lmin"]) ** (k / max(1, m - 1))))
        off, C = _aniso(L, es[k])
        out.append((off, C, _rand(seed, 100 + k, L * L)))
    return out


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("spmv", "graph", "spmm"):
        P.psb_spmm(1.0, s["a"], s["x"], 0.0, s["y"], trans=case.get("trans", "N"))
        return s["ty"]
    if kind == "spsm":
        P.psb_spsm(1.0, s["a"], s["x"], 0.0, s["y"], trans=case["trans"])
        return s["ty"]
    if kind == "vector":
        # the vector operations of one preconditioned CG step
        P.psb_geaxpbyz(0.7, s["p"], 1.0, s["q"], s["x"])       # x = x + alpha p
        P.psb_geaxpbyz(-0.3, s["q"], 1.0, s["r"], s["y"])      # r = r - alpha q
        P.psb_gemlt(1.0, s["d"], s["y"], 0.0, s["z"])          # z = D r
        rz = P.psb_gedot(s["y"], s["z"])
        rr = P.psb_genrm2(s["y"])
        return {"x": s["tx"], "y": s["ty"], "z": s["tz"], "rz": rz, "rr": rr}
    if kind == "krylov":
        P.psb_geaxpby(0.0, s["b"], 0.0, s["x"])
        P.psb_krylov(case["method"], s["a"], s["prec"], s["b"], s["x"], 1e-10, s["desc"],
                     itmax=2000)
        return s["tx"]
    if kind == "fused":
        P.psb_geaxpby(0.0, s["b"], 0.0, s["x"])
        if case["mixed"]:
            P.psb_krylov_mixed(case["method"], s["a"], s["prec"], s["b"], s["x"], 1e-10, s["desc"],
                               variant="reliable")
        else:
            P.psb_krylov_fused(case["method"], s["a"], s["prec"], s["b"], s["x"], 1e-10, s["desc"],
                               itmax=2000)
        return s["tx"]
    s["eng"].solve(s["jobs"], eps=1e-8, itmax=20000)
    return s["tx"]


# ------------------------------------------------------------------ what it takes
def _its(method, prec, L):
    """Iterations a solve to 1e-10 takes, roughly."""
    if method == "RGMRES":
        return 0.07 * L * L
    per = {"CG": 3.0, "BICGSTAB": 2.5}[method]
    return per * L * (0.4 if prec == "BJAC" else 1.0)


def work(case):
    kind = case["kind"]
    es = 4 if case.get("dtype") == "s" else 8
    if kind == "graph":
        n, nnz = case["n"], 16 * case["n"]
        return {"bytes": (2 * es + 4) * n + (es + 4) * nnz, "flops": 2 * nnz}
    if kind == "vector":
        return {"bytes": 3 * 3 * es * case["n"], "flops": 9 * case["n"]}
    if kind == "batch":
        b = f = 0
        for k in range(case["nsys"]):
            L = case["lmin"] * (case["lmax"] / case["lmin"]) ** (k / max(1, case["nsys"] - 1))
            its = 2.5 * L
            # FP32: values and indices of 5 entries a row, 12 vector passes
            b += its * L * L * (5 * 8 + 12 * 4)
            f += its * L * L * (2 * 5 + 12)
        return {"bytes": b, "flops": f}
    L = case["L"]
    n = L ** 3
    nnz = 7 * n - 6 * L * L
    if kind == "spmv":
        return {"bytes": (2 * es + 4) * n + (es + 4) * nnz, "flops": 2 * nnz}
    if kind == "spmm":
        k = case["k"]
        return {"bytes": 4 * n + (es + 4) * nnz + 2 * es * n * k, "flops": 2 * nnz * k}
    if kind == "spsm":
        tri = (nnz - n) // 2 + n
        return {"bytes": (2 * es + 4) * n + (es + 4) * tri, "flops": 2 * tri}
    its = _its(case["method"], case.get("prec", "DIAG"), L)
    es = 4 if case.get("mixed") else 8
    two = 2 if case["method"] == "BICGSTAB" else 1
    mat = (es + 4) * nnz + (2 * es + 4) * n
    if case.get("prec") == "BJAC":
        mat += 12 * nnz + 24 * n
    return {"bytes": its * (two * mat + 12 * two * es * n), "flops": its * two * (2 * nnz + 10 * n)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("spmv", "graph", "spmm", "spsm", "vector"):
        # sums of a row or vector in another order, in the case's precision
        # (against 64 bits: up to 2e-7 seen in FP32, 6e-16 in FP64)
        return {"rel": 2e-6 if case["dtype"] == "s" else 1e-14}
    # whole solves stop on a residual of 1e-10 (1e-8 in the batch), some
    # condition number away from the solution (2e-8 and 4e-6 seen)
    return {"rel": 2e-5 if kind == "batch" else 2e-7}


# ------------------------------------------------------------------ in 64 bits
def _levels_solve(off, C, x, lower, L):
    """T^-1 x for a triangle in _stencil's form, plane of equal x+y+z after plane."""
    n = C.shape[1]
    r = torch.arange(n, device=DEV)
    lev = r % L + (r // L) % L + r // (L * L)
    order = torch.argsort(lev, stable=True)
    ptr = torch.cumsum(torch.bincount(lev, minlength=3 * L - 2), 0).tolist()
    ptr = [0] + ptr
    y = torch.zeros_like(x)
    steps = range(3 * L - 2) if lower else reversed(range(3 * L - 2))
    ks = [k for k, o in enumerate(off) if (o < 0 if lower else o > 0)]
    d = C[off.index(0)]
    for v in steps:
        i = order[ptr[v]:ptr[v + 1]]
        acc = x[i].clone()
        for k in ks:
            acc -= C[k][i] * y[(i + off[k]).clamp(0, n - 1)]
        y[i] = acc / d[i]
    return y


def exact(case, seed):
    kind, single = case["kind"], case.get("dtype") == "s"
    if kind in ("spmv", "spmm", "spsm"):
        off, C = _stencil(case["L"], seed, single=single)
        n = C.shape[1]
        if kind == "spmm":
            return _apply(off, C, _rand(seed, 1, n, case["k"], single=single)).T.contiguous()
        x = _rand(seed, 1, n, single=single)
        if kind == "spmv":
            return _apply(*(_transposed(off, C) if case["trans"] == "T" else (off, C)), x)
        lower = case["lower"]
        if case["trans"] == "T":
            off, C = _transposed(off, C)
            lower = not lower
        return _levels_solve(off, C, x, lower, case["L"])
    if kind == "graph":
        ia, ja, val = _graph(case["n"], seed, single)
        x = _rand(seed, 1, case["n"], single=single)
        return torch.zeros_like(x).index_add_(0, ia, val * x[ja])
    if kind == "vector":
        p, q, r, d = (_vector_input(case, seed, j) for j in range(4))
        alpha, beta = 0.7, -0.3
        if single:
            alpha, beta = float(np.float32(alpha)), float(np.float32(beta))
        y = r + beta * q
        z = d * y
        return {"x": q + alpha * p, "y": y, "z": z, "rz": float(torch.dot(y, z)),
                "rr": float(torch.linalg.vector_norm(y))}
    if kind == "batch":
        return [xt for _, _, xt in _systems(case, seed)]
    return _rand(seed, 1, case["L"] ** 3)
