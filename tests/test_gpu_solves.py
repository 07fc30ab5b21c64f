"""GPU: the triangular solves where a front changes kind and a right-hand side changes path.

Few columns are solved one by one, more in blocks of sixteen; small fronts are grouped four to a
task, a front of one diagonal block and at most four row blocks is one task, longer ones are
chains, and separators of more than eight tiles are products of their own.  Every size pair lies
at one of these lines; every number of columns is compared with the dense solution."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

# (block, separator): fronts of nn = block, na = separator, and a root of nn = separator
SIZES = [(1, 1), (16, 16), (17, 47), (20, 44), (20, 45), (31, 33), (33, 31), (64, 1), (64, 64), (40, 65), (64, 255),
         (64, 256), (64, 257), (65, 256), (15, 512), (17, 513), (33, 576), (129, 520), (200, 1030)]
COLS = [1, 2, 3, 4, 5, 6, 15, 16, 17, 33]


def _dense(nb, ns, blocks, seed, indefinite):
    rng = np.random.default_rng(seed)
    n = blocks * nb + ns
    A = np.zeros((n, n))
    for k in range(blocks):
        A[k * nb:(k + 1) * nb, k * nb:(k + 1) * nb] = rng.uniform(-1, 1, (nb, nb))
    A[blocks * nb:, :] = rng.uniform(-1, 1, (ns, n))
    A = np.tril(A, -1)
    A = A + A.T
    d = np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)  # diagonally dominant
    if indefinite:
        d *= np.where(rng.random(n) < 0.3, -1.0, 1.0)
    return A + np.diag(d)


def _check(ct, A, ldlt, f32, cols, seed):
    n = A.shape[0]
    C = sp.csc_matrix(A)
    P, S = ct.symbolic(C)
    prec = ct.MF_FP32 if f32 else ct.MF_FP64
    F = ct.ldlt_(ct.ChordalLDLt(C, P, S, precision=prec)) if ldlt else ct.cholesky_(ct.ChordalCholesky(C, P, S, precision=prec))
    assert ct.issuccess(F)
    B = np.random.default_rng(seed).standard_normal((n, max(cols)))
    ref = np.linalg.solve(A, B)
    # diagonally dominant (condition number of order one after scaling): n eps, with the margin
    # of the tile tests (1e-12 in FP64, 1e-4 in FP32)
    tol = 1e-4 if f32 else 1e-12
    for k in cols:
        X = ct.solve(F, B[:, :k])
        err = np.linalg.norm(X - ref[:, :k], axis=0) / np.linalg.norm(ref[:, :k], axis=0)
        assert err.max() <= tol, (k, err.max())
    x = ct.solve(F, B[:, 0])
    assert np.linalg.norm(x - ref[:, 0]) <= tol * np.linalg.norm(ref[:, 0])


@pytest.mark.parametrize("nb,ns", SIZES)
@pytest.mark.parametrize("kind", ["chol", "ldlt", "chol_f32"])
def test_front_sizes(ct, nb, ns, kind):
    print(kind, nb, ns, flush=True)
    ldlt = kind == "ldlt"
    _check(ct, _dense(nb, ns, 2, 100 * nb + ns, ldlt), ldlt, kind == "chol_f32", COLS, nb + ns)


@pytest.mark.parametrize("nb,ns,kids", [(2, 20, 33), (5, 70, 21), (30, 20, 9), (3, 300, 40), (66, 130, 5)])
def test_many_children(ct, nb, ns, kids):
    """A parent with fewer and more children than it gathers at a time, small fronts that fill
    their groups by count (nb = 2) and by size (nb = 30)."""
    print(nb, ns, kids, flush=True)
    for ldlt in (False, True):
        _check(ct, _dense(nb, ns, kids, kids, ldlt), ldlt, False, [1, 4, 16, 20], 3)


def test_nonfinite_columns_stay_apart(ct):
    """An infinity or a NaN in one right-hand side ends the solve and leaves the others as they
    were (every wait ends: a value that is not a number is a value)."""
    A = _dense(70, 90, 2, 7, False)
    C = sp.csc_matrix(A)
    P, S = ct.symbolic(C)
    F = ct.cholesky_(ct.ChordalCholesky(C, P, S))
    n = A.shape[0]
    B = np.random.default_rng(1).standard_normal((n, 4))
    good = ct.solve(F, B)
    # a quiet NaN, an infinity, and signalling NaNs of both halves of the payload range
    odd = np.array([np.nan, np.inf, 0.0, 0.0])
    odd[2:] = np.array([0x7FF4A5A5DEADBEE1, 0x7FF0000000000001], dtype=np.uint64).view(np.float64)
    for v in odd:
        for row in (0, 69, 150, n - 1):
            D = B.copy()
            D[row, 1] = v
            X = ct.solve(F, D)
            assert not np.isfinite(X[:, 1]).all()
            assert np.array_equal(X[:, [0, 2, 3]], good[:, [0, 2, 3]])


@pytest.mark.parametrize("cols", [5, 6, "half", "most"])
def test_fixed_scratch(ct, cols):
    """The solve without allocation from few columns up to as many as its fixed array takes: the
    blocked form while its workspaces fit, a few columns at a time up to the limit, refused past it."""
    import ctypes
    import torch
    from cliquetrees_amd import _native
    lib = _native.hip()
    pr = ct.problems
    A = pr.laplacian3d_7pt(14, 12, 11, seed=3)
    P, S = ct.symbolic(A, alg=ct.grid_nd(14, 12, 11))
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S))
    n, h = A.shape[0], F._f.handle
    perm = np.ascontiguousarray(P.perm, dtype=np.int64)
    pp = perm.ctypes.data_as(_native.i64p)

    def call(X, k):
        return lib.mf_solve_noalloc(h, pp, ctypes.c_void_p(X.data_ptr() if X is not None else 16), k, n)

    # the first column count that is refused (the call returns before anything is enqueued)
    st = np.zeros(23, np.int64)
    lib.mf_plan_stats(F._f.plan.handle, st.ctypes.data_as(_native.i64p), 23)
    most = (64 << 20) // (8 * (n + int(st[22])))
    while ((8 * int(st[22]) * most + 255) // 256 * 256) + 8 * n * most > 64 << 20:
        most -= 1
    k = {"half": most // 2, "most": most}.get(cols, cols)
    print(cols, k, most, flush=True)
    B = torch.tensor(np.random.default_rng(1).standard_normal((k, n)), device="cuda")
    X = B.clone()
    assert call(X, k) == 0, lib.mf_last_error()
    assert lib.mf_factor_sync(h) == 0
    torch.cuda.synchronize()
    x, b = X.cpu().numpy().T, B.cpu().numpy().T
    # n eps (condition number of the grid of order n): 1e-10
    assert np.linalg.norm(A @ x - b) <= 1e-10 * np.linalg.norm(b)
    assert call(None, most + 1) == -1 and b"scratch" in lib.mf_last_error()
