"""Workloads of the multifrontal engine, one pass each through its public entry points.

Every case is a dict with a ``kind`` and the sizes of one input:

  step      device-resident values -> value refresh, Cholesky factorization
            and a solve (the loop of an implicit time stepper or a Newton
            iteration on a fixed pattern)
  mixed     the same with FP32 fronts and FP64 iterative refinement
  solve     a solve with a factor that is already on the device
  batch     many small systems of uneven size as one forest, one right-hand
            side each
  kkt       one request of the serving loop: LDLt of a quasi-definite KKT
            matrix and a solve with one FP64 correction
  selinv    selected inversion of a resident factor, read out in the
            reference layout
  dropin    ``chol_impl!`` on host arrays, as the reference's own API calls it
  complete  ``complete_impl!`` on host arrays

Patterns are analysed once and kept, as every user of the engine does:
``prepare`` makes new values and right-hand sides from the seed.
"""
from __future__ import annotations

import ctypes
import functools
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its directory name is not an identifier)."""
    if "cliquetrees_amd" not in sys.modules:
        pkg = os.path.join(ROOT, "cliquetrees.jl_amd")
        spec = importlib.util.spec_from_file_location("cliquetrees_amd", os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["cliquetrees_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["cliquetrees_amd"]


ct = _package()
from cliquetrees_amd import _native  # noqa: E402


def listed():
    return [
        # the smallest call: a 2-D Dirichlet grid in minimum-degree order, one
        # right-hand side; the chain of tiny fronts and the launches count
        {"name": "step_2d_100_mmd", "kind": "step", "grid": "2d", "nx": 100, "ny": 100, "nz": 1,
         "order": "mmd", "nrhs": 1},
        # an ordinary 3-D grid with odd edges and a few right-hand sides
        {"name": "step_3d_31x29x27", "kind": "step", "grid": "7pt", "nx": 31, "ny": 29, "nz": 27,
         "order": "nd", "nrhs": 3},
        # the headline: 64^3 7-point Laplacian, 16 right-hand sides, FP64
        {"name": "step_3d_64", "kind": "step", "grid": "7pt", "nx": 64, "ny": 64, "nz": 64,
         "order": "nd", "nrhs": 16},
        # denser rows and wider fronts for the same number of unknowns
        {"name": "step_27pt_48", "kind": "step", "grid": "27pt", "nx": 48, "ny": 48, "nz": 48,
         "order": "nd", "nrhs": 16},
        # FP32 fronts, FP64 refinement to full accuracy
        {"name": "mixed_27pt_40x36x44", "kind": "mixed", "grid": "27pt", "nx": 40, "ny": 36, "nz": 44,
         "order": "nd", "nrhs": 16},
        # a large resident factor and a single right-hand side
        {"name": "solve_3d_56x60x52_1", "kind": "solve", "grid": "7pt", "nx": 56, "ny": 60, "nz": 52,
         "order": "nd", "nrhs": 1},
        # a mid-sized factor and a block of right-hand sides of odd width
        {"name": "solve_3d_40_75", "kind": "solve", "grid": "7pt", "nx": 40, "ny": 40, "nz": 40,
         "order": "nd", "nrhs": 75},
        # uneven systems of 50..2000 unknowns, half 2-D and half 3-D
        {"name": "batch_600", "kind": "batch", "count": 600},
        # a serving request of the KKT stream
        {"name": "kkt_7000", "kind": "kkt", "nh": 7000, "signs": False},
        # marginal variances of a 3-D Gaussian field
        {"name": "selinv_3d_28x30x26", "kind": "selinv", "grid": "7pt", "nx": 28, "ny": 30, "nz": 26,
         "order": "nd"},
        # the reference's own call on host arrays, copies included
        {"name": "dropin_3d_26x28x25", "kind": "dropin", "grid": "7pt", "nx": 26, "ny": 28, "nz": 25,
         "order": "nd", "uplo": "L"},
        # maximum-determinant completion of a covariance on a chordal pattern
        {"name": "complete_3d_18x20x17", "kind": "complete", "grid": "7pt", "nx": 18, "ny": 20, "nz": 17,
         "order": "nd", "uplo": "L"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims3(rng, nmin, nmax):
    """A box of about n unknowns, n log-uniform, edges within a third of each other."""
    n = math.exp(rng.uniform(math.log(nmin), math.log(nmax)))
    a = n ** (1 / 3)
    nx, ny = (max(4, int(round(a * rng.uniform(0.82, 1.2)))) for _ in range(2))
    return nx, ny, max(4, int(round(n / (nx * ny))))


def draw(rng):
    """A case of the ranges that the listed ones stand for (none costs more than the largest of them)."""
    kind = rng.choice(["step", "step", "step", "mixed", "solve", "solve", "batch", "kkt", "selinv", "dropin",
                       "complete"])
    if kind == "batch":
        return {"kind": kind, "count": _log_int(rng, 20, 800)}
    if kind == "kkt":
        return {"kind": kind, "nh": _log_int(rng, 1000, 9000), "signs": rng.random() < 0.5}
    if kind == "step" and rng.random() < 0.35:
        nx, ny = _log_int(rng, 25, 320), _log_int(rng, 25, 320)
        return {"kind": kind, "grid": "2d", "nx": nx, "ny": ny, "nz": 1, "order": rng.choice(["nd", "mmd"]),
                "nrhs": _log_int(rng, 1, 33)}
    grid = "7pt" if kind in ("selinv", "dropin", "complete") else rng.choice(["7pt", "27pt"])
    top = {"step": 200000, "mixed": 120000, "solve": 200000, "selinv": 30000, "dropin": 25000,
           "complete": 7000}[kind]
    if grid == "27pt":
        top = min(top, 95000)
    nx, ny, nz = _dims3(rng, 700, top)
    c = {"kind": kind, "grid": grid, "nx": nx, "ny": ny, "nz": nz, "order": "nd"}
    if kind in ("step", "mixed", "solve"):
        c["nrhs"] = _log_int(rng, 1, 40 if kind != "solve" else 90)
    if kind in ("dropin", "complete"):
        c["uplo"] = rng.choice(["L", "U"])
    return c


# ---- patterns (analysed once) and values (from the seed) ---------------------------------


class _Pattern:
    """A matrix pattern, its analysis, and what turns edge weights into values."""

    def __init__(self, A, order, sizes=None):
        A.sort_indices()
        self.A, self.n, self.nnz = A, A.shape[0], int(A.nnz)
        self.P, self.S = ct.symbolic(A, alg=order)
        self.flat = {}
        self.perm = np.ascontiguousarray(self.P.perm, dtype=np.int64)
        self.sizes = sizes
        rows = A.indices.astype(np.int64)
        cols = np.repeat(np.arange(self.n, dtype=np.int64), np.diff(A.indptr))
        self.rows, self.cols = rows, cols
        off = np.nonzero(rows != cols)[0]
        self.off, self.dia = off, np.nonzero(rows == cols)[0]
        key = np.minimum(rows[off], cols[off]) * self.n + np.maximum(rows[off], cols[off])
        edges, self.eid = np.unique(key, return_inverse=True)
        self.lo, self.hi = edges // self.n, edges % self.n

    def flat_of(self, uplo):
        if uplo not in self.flat:
            self.flat[uplo] = ct.flatindices(self.S, self.A, uplo)
        return self.flat[uplo]

    def plan(self):
        return ct.device_plan(self.S)

    def laplacian_values(self, seed, shift=1e-3):
        """Graph Laplacian of U[0.5, 1.5] edge weights plus shift I, in the pattern's CSC order."""
        w = np.random.default_rng(seed).uniform(0.5, 1.5, size=len(self.lo))
        deg = np.bincount(self.lo, w, self.n) + np.bincount(self.hi, w, self.n) + shift
        v = np.empty(self.nnz)
        v[self.off] = -w[self.eid]
        v[self.dia] = deg[self.rows[self.dia]]
        return v


@functools.lru_cache(maxsize=6)
def _grid(grid, nx, ny, nz, order):
    if grid == "2d":
        A = ct.problems.grid_laplacian_random((nx, ny), 0)
    elif grid == "7pt":
        A = ct.problems.laplacian3d_7pt(nx, ny, nz, 0)
    else:
        A = ct.problems.stencil3d_27pt(nx, ny, nz, 0)
    return _Pattern(A, "mmd" if order == "mmd" else ct.grid_nd(nx, ny, nz))


@functools.lru_cache(maxsize=2)
def _batch(count):
    """The systems of a batch as BatchedFactorization lays them out: one forest."""
    specs = ct.problems.batch_specs(count, 4)
    mats = [ct.problems.grid_laplacian_random(d, 0) for d in specs]
    orders = [ct.grid_nd(*(d if len(d) == 3 else (d[0], d[1], 1))) for d in specs]
    sizes = np.array([m.shape[0] for m in mats], dtype=np.int64)
    offs = np.concatenate([[0], np.cumsum(sizes)])
    colptr = np.concatenate([[0]] + [m.indptr[1:].astype(np.int64) for m in mats])
    base = np.cumsum([0] + [m.nnz for m in mats])
    colptr[1:] += np.repeat(base[:-1], sizes)
    rows = np.concatenate([m.indices.astype(np.int64) + o for m, o in zip(mats, offs)])
    data = np.concatenate([m.data for m in mats])
    A = type(mats[0])((data, rows, colptr), shape=(int(offs[-1]),) * 2)
    return _Pattern(A, np.concatenate([o + off for o, off in zip(orders, offs)]), sizes)


@functools.lru_cache(maxsize=2)
def _kkt(nh):
    K, nh, m = ct.problems.kkt_matrix(ct.problems.near_cubic_dims(nh, 3), seed=500)
    p = _Pattern(K, "mmd")
    p.nh, p.base = nh, np.array(K.data)
    return p


def _pattern(case):
    if case["kind"] == "batch":
        return _batch(case["count"])
    if case["kind"] == "kkt":
        return _kkt(case["nh"])
    return _grid(case["grid"], case["nx"], case["ny"], case["nz"], case["order"])


def _values(case, p, seed):
    if case["kind"] == "kkt":  # a value update of the stream: the Hessian's diagonal rescaled
        v = p.base.copy()
        d = p.dia[p.rows[p.dia] < p.nh]
        v[d] *= np.random.default_rng(seed).uniform(0.1, 10.0, size=len(d))
        return v
    return p.laplacian_values(seed)


def _rhs(case, p, seed):
    """nrhs x n (column-major n x nrhs), N(0, 1)."""
    return np.random.default_rng(seed + 7777777).standard_normal((case.get("nrhs", 1), p.n))


def _covariance(case, p, seed):
    """An exponential covariance with uneven variances on the factor's pattern, reference layout."""
    rng = np.random.default_rng(seed)
    sd, ell = rng.uniform(0.5, 2.0, size=p.n), rng.uniform(2.0, 6.0)
    x = np.stack([np.arange(p.n) % case["nx"], np.arange(p.n) // case["nx"] % case["ny"],
                  np.arange(p.n) // (case["nx"] * case["ny"])], 1).astype(np.float64)
    x, sd = x[p.perm - 1], sd[p.perm - 1]

    def cov(i, j):
        return sd[i] * sd[j] * np.exp(-np.sqrt(((x[i] - x[j]) ** 2).sum(1)) / ell)

    (ri, ci), (rl, cl) = _layout(p, case["uplo"])
    D = np.zeros(len(ri))
    low = ri >= ci if case["uplo"] == "L" else ri <= ci
    D[low] = cov(ri[low], ci[low])
    return D, cov(rl, cl)


def _layout(p, uplo):
    """0-based (row, column) in the permuted order of every slot of Dval and of Lval."""
    key = "layout" + uplo
    if key not in p.flat:
        S = p.S
        dr, dc, lr, lc = [], [], [], []
        for j in range(S.nfr):
            res = np.arange(S.resptr[j] - 1, S.resptr[j + 1] - 1)
            sep = S.septgt[S.sepptr[j] - 1:S.sepptr[j + 1] - 1] - 1
            r, c = np.tile(res, len(res)), np.repeat(res, len(res))
            dr.append(r)
            dc.append(c)
            if uplo == "L":
                lr.append(np.tile(sep, len(res)))
                lc.append(np.repeat(res, len(sep)))
            else:
                lr.append(np.tile(res, len(sep)))
                lc.append(np.repeat(sep, len(res)))
        p.flat[key] = ((np.concatenate(dr), np.concatenate(dc)), (np.concatenate(lr), np.concatenate(lc)))
    return p.flat[key]


@functools.lru_cache(maxsize=1)
def _stream():
    """The program's compute stream, shared by torch and the engine."""
    return torch.cuda.Stream()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _ok(rc):
    if rc != 0:
        raise RuntimeError(_native.hip().mf_last_error())


class _State:
    pass


def prepare(case, seed):
    p = _pattern(case)
    s = _State()
    s.case, s.p, s.kind, s.lib = case, p, case["kind"], _native.hip()
    if s.kind in ("dropin", "complete"):
        # host arrays, as the reference holds them
        if s.kind == "complete":
            s.D, s.L = _covariance(case, p, seed)
        else:
            v = np.concatenate([[0.0], _values(case, p, seed)])
            flat = p.flat_of(case["uplo"])
            full = np.zeros(p.S.ndz + p.S.nlz + 1)
            full[flat] = v[1:]
            s.D, s.L = full[1:p.S.ndz + 1].copy(), full[p.S.ndz + 1:].copy()
        p.plan()
        return s
    s.diag = ct.MF_LDLT if s.kind == "kkt" else ct.MF_CHOLESKY
    s.fac = ct.DeviceFactor(p.plan(), ct.MF_FP32 if s.kind == "mixed" else ct.MF_FP64)
    s.h = s.fac.handle
    flat = p.flat_of("L")
    _ok(s.lib.mf_factor_set_pattern(s.h, len(flat), flat.ctypes.data_as(_native.i64p)))
    s.stream = _stream()
    _ok(s.lib.mf_factor_set_stream(s.h, ctypes.c_void_p(s.stream.cuda_stream)))
    s.perm = p.perm.ctypes.data_as(_native.i64p)
    s.vals = torch.tensor(_values(case, p, seed), dtype=torch.float64, device="cuda")
    s.nrhs = case.get("nrhs", 1)
    if s.kind != "selinv":
        s.B = torch.tensor(_rhs(case, p, seed), dtype=torch.float64, device="cuda")
        s.X = torch.empty_like(s.B)
    if s.kind in ("mixed", "kkt"):
        cp = np.ascontiguousarray(p.A.indptr, dtype=np.int64) + 1
        rv = np.ascontiguousarray(p.A.indices, dtype=np.int64) + 1
        _ok(s.lib.mf_factor_set_matrix(s.h, p.n, cp.ctypes.data_as(_native.i64p), rv.ctypes.data_as(_native.i64p),
                                       _ptr(s.vals), 1))
        s.seg = np.array([0, p.n], dtype=np.int64)
    if s.kind == "kkt":
        s.nrm = torch.empty(2, dtype=torch.float64, device="cuda")
        s.signs = None
        if case["signs"]:
            sg = np.where(np.arange(p.n) < p.nh, 1.0, -1.0)[p.perm - 1]
            s.signs = torch.tensor(sg, dtype=torch.float64, device="cuda")
    if s.kind == "selinv":
        s.D = torch.empty(p.S.ndz, dtype=torch.float64, device="cuda")
        s.L = torch.empty(p.S.nlz, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    if s.kind in ("solve", "selinv"):
        _factorize(s)
        info = ctypes.c_int64(0)
        _ok(s.lib.mf_factor_info(s.h, ctypes.byref(info)))
        assert info.value == 0
    return s


def _factorize(s):
    _ok(s.lib.mf_factor_refresh(s.h, _ptr(s.vals), 1))
    signs = _ptr(s.signs) if s.kind == "kkt" and s.signs is not None else None
    _ok(s.lib.mf_factorize_async(s.h, s.diag, signs, 0, 0.0, 0.0))


def run(s):
    n = s.p.n
    if s.kind == "dropin":
        D, L, _, info = ct.chol_impl(s.p.S, s.D, s.L, uplo=s.case["uplo"])
        return {"D": D, "L": L, "info": info}
    if s.kind == "complete":
        D, L, info = ct.complete_impl(s.p.S, s.D, s.L, uplo=s.case["uplo"])
        return {"D": D, "L": L, "info": info}
    if s.kind == "selinv":
        _ok(s.lib.mf_selinv(s.h))
        _ok(s.lib.mf_selinv_get(s.h, _ptr(s.D), _ptr(s.L), 1))
        return {"D": s.D, "L": s.L}
    if s.kind != "solve":
        _factorize(s)
    if s.kind == "mixed":
        it, rr = ctypes.c_int(0), ctypes.c_double(0.0)
        _ok(s.lib.mf_refine(s.h, s.perm, _ptr(s.B), n, _ptr(s.X), n, s.nrhs, 1, 1e-12, 20, ctypes.byref(it),
                            ctypes.byref(rr)))
    elif s.kind == "kkt":
        _ok(s.lib.mf_refine_steps(s.h, s.perm, _ptr(s.B), n, _ptr(s.X), n, s.nrhs, 1, 1,
                                  s.seg.ctypes.data_as(_native.i64p), _ptr(s.nrm)))
    else:
        with torch.cuda.stream(s.stream):
            s.X.copy_(s.B, non_blocking=True)
        _ok(s.lib.mf_solve(s.h, s.perm, _ptr(s.X), s.nrhs, n, 1))
    return {"X": s.X}


def work(case):
    """Flops of the reference's own fronts; A's values in, the factor and the results moved once."""
    p = _pattern(case)
    S, kind = p.S, case["kind"]
    nn, na = S.nn().astype(np.float64), S.na().astype(np.float64)
    factor = 8.0 * float((nn * (nn + 1) / 2 + nn * na).sum())
    chol = S.factor_flops()
    nrhs = case.get("nrhs", 1)
    vec = 16.0 * p.n * nrhs
    if kind == "step" or kind == "batch":
        return {"bytes": 8.0 * p.nnz + factor + vec, "flops": chol + S.solve_flops(nrhs)}
    if kind == "mixed":
        return {"bytes": 8.0 * p.nnz + factor / 2 + vec, "flops": chol + S.solve_flops(nrhs)}
    if kind == "kkt":
        return {"bytes": 8.0 * p.nnz + factor + vec, "flops": chol + 2 * S.solve_flops(nrhs)}
    if kind == "solve":
        return {"bytes": factor + vec, "flops": S.solve_flops(nrhs)}
    if kind == "selinv":
        return {"bytes": 2 * factor, "flops": float((2 * na * na * nn + 2 * na * nn * nn + 2 * nn ** 3 / 3).sum())}
    if kind == "dropin":
        return {"bytes": 2 * factor, "flops": chol}
    return {"bytes": 2 * factor,
            "flops": float((na ** 3 / 3 + 2 * na * na * nn + 2 * na * nn * nn + 2 * nn ** 3 / 3).sum())}


# ---- the same results in plain 64-bit torch / numpy ------------------------------------------


def _cg(p, v, B):
    """A X = B by conjugate gradients on the device, then corrected from the true residual."""
    dev = torch.device("cuda")
    deg = np.diff(p.A.indptr)
    width = int(deg.max())
    col = np.zeros((width, p.n), dtype=np.int64)
    val = np.zeros((width, p.n))
    slot = np.arange(p.nnz) - np.repeat(p.A.indptr[:-1].astype(np.int64), deg)
    col[slot, p.cols], val[slot, p.cols] = p.rows, v  # the matrix is symmetric
    col, val = torch.tensor(col, device=dev), torch.tensor(val, device=dev)
    dinv = torch.tensor(1.0 / v[p.dia], device=dev)[:, None]

    def mul(x):
        y = val[0][:, None] * x[col[0]]
        for k in range(1, width):
            y += val[k][:, None] * x[col[k]]
        return y

    b = torch.tensor(B, device=dev).T.contiguous()
    x = torch.zeros_like(b)
    for _ in range(3):
        r = b - mul(x)
        z = dinv * r
        d, rz, stop = z.clone(), (r * z).sum(0), None
        y = torch.zeros_like(b)
        for k in range(4000):
            q = mul(d)
            a = rz / (d * q).sum(0).clamp_min(1e-300)
            y += a * d
            r -= a * q
            z = dinv * r
            rz2 = (r * z).sum(0)
            d = z + (rz2 / rz.clamp_min(1e-300)) * d
            rz = rz2
            if k % 50 == 0:
                if stop is None:
                    stop = 1e-24 * float(rz.max())
                if float(rz.max()) <= stop:
                    break
        x += y
    return x.T.contiguous()


def _dense(p, v, permuted):
    i, j = p.rows, p.cols
    if permuted:
        i, j = p.P.invp[i] - 1, p.P.invp[j] - 1
    A = torch.zeros((p.n, p.n), dtype=torch.float64, device="cuda")
    A[torch.tensor(i, device="cuda"), torch.tensor(j, device="cuda")] = torch.tensor(v, device="cuda")
    return A


def _tri_inverse(L):
    """Inverse of a lower triangular matrix by halves, in place."""
    n = L.shape[0]
    if n <= 512:
        L.copy_(torch.linalg.solve_triangular(L, torch.eye(n, dtype=L.dtype, device=L.device), upper=False))
        return L
    h = n // 2
    _tri_inverse(L[:h, :h])
    _tri_inverse(L[h:, h:])
    L[h:, :h] = -(L[h:, h:] @ (L[h:, :h] @ L[:h, :h]))
    return L


def _slots(p, M, uplo, low):
    """Dval and Lval of a dense permuted matrix (its lower triangle)."""
    out = []
    for k, (r, c) in enumerate(_layout(p, uplo)):
        i, j = torch.tensor(np.maximum(r, c), device="cuda"), torch.tensor(np.minimum(r, c), device="cuda")
        x = M[i, j]
        if k == 0 and low:
            x[torch.tensor(r < c if uplo == "L" else r > c, device="cuda")] = 0.0
        out.append(x)
    return out


def exact(case, seed):
    p, kind = _pattern(case), case["kind"]
    if kind == "complete":
        return _complete_exact(case, p, seed)
    v = _values(case, p, seed)
    if kind in ("selinv", "dropin"):
        if p.n > 32000:
            return None
        A = _dense(p, v, True)
        A = torch.linalg.cholesky(A)
        if kind == "dropin":
            D, L = _slots(p, A, case["uplo"], True)
            return {"D": D.cpu().numpy(), "L": L.cpu().numpy(), "info": None}
        A = _tri_inverse(A.tril_())
        inv = A.T @ A
        D, L = _slots(p, inv, "L", True)
        return {"D": D, "L": L}
    B = _rhs(case, p, seed)
    if kind == "kkt":
        A = _dense(p, v, False)
        b = torch.tensor(B, device="cuda").T.contiguous()
        lu, piv = torch.linalg.lu_factor(A)
        x = torch.linalg.lu_solve(lu, piv, b)
        for _ in range(3):
            x += torch.linalg.lu_solve(lu, piv, b - A @ x)
        return {"X": x.T.contiguous()}
    return {"X": _cg(p, v, B)}


def _complete_exact(case, p, seed):
    """Per clique, with M = Sigma(sep, sep): D D' = (Sigma11 - Sigma12 M^-1 Sigma21)^-1, D lower
    triangular, and L21 = -M^-1 Sigma21 D."""
    uplo = case["uplo"]
    D, L = _covariance(case, p, seed)
    S = p.S
    key = []
    for (r, c) in _layout(p, uplo):
        key.append(np.maximum(r, c) * p.n + np.minimum(r, c))
    key = np.concatenate(key)
    val = np.concatenate([D, L])
    r, c = _layout(p, uplo)[0]
    keep = np.ones(len(key), dtype=bool)
    keep[:len(D)] = r >= c if uplo == "L" else r <= c
    order = np.argsort(key[keep], kind="stable")
    key, val = key[keep][order], val[keep][order]

    def block(i, j):
        a, b = np.meshgrid(i, j, indexing="ij")
        return val[np.searchsorted(key, np.maximum(a, b) * p.n + np.minimum(a, b))]

    D2, L2 = np.zeros_like(D), np.zeros_like(L)
    for j in range(S.nfr):
        res = np.arange(S.resptr[j] - 1, S.resptr[j + 1] - 1)
        sep = S.septgt[S.sepptr[j] - 1:S.sepptr[j + 1] - 1] - 1
        C = block(res, res)
        if len(sep):
            X = np.linalg.solve(block(sep, sep), block(sep, res))
            C = C - block(res, sep) @ X
        # C^-1 = D D' with D lower triangular: reversing rows and columns turns
        # C = (D')^-1 D^-1 into an ordinary Cholesky factorization
        R = np.linalg.cholesky(C[::-1, ::-1])
        Dj = np.tril(np.linalg.inv(R)[::-1, ::-1].T)
        nn, na = len(res), len(sep)
        D2[S.Dptr[j] - 1:S.Dptr[j] - 1 + nn * nn] = (Dj if uplo == "L" else Dj.T).ravel(order="F")
        if na:
            Lj = -X @ Dj
            L2[S.Lptr[j] - 1:S.Lptr[j] - 1 + na * nn] = (Lj if uplo == "L" else Lj.T).ravel(order="F")
    return {"D": D2, "L": L2, "info": None}
