"""GPU: infinite and subnormal pivots of the small fronts (one wavefront up to nJ = 32, one
workgroup up to 64), against the oracle.  An infinite diagonal entry pins its unknown: the
multipliers below it are zero and every other column is that of the matrix without the unknown."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _matrix(n, kids, seed):
    """`kids` dense blocks of n - 8 columns, each coupled to the same 8 columns."""
    rng = np.random.default_rng(seed)
    c = n - 8
    N = kids * c + 8
    A = np.zeros((N, N))
    for k in range(kids):
        A[k * c:(k + 1) * c, k * c:(k + 1) * c] = rng.uniform(-1, 1, (c, c))
    A[kids * c:, :] = rng.uniform(-1, 1, (8, N))
    A = np.tril(A, -1)
    A = A + A.T
    return A + np.diag(np.abs(A).sum(1) + rng.uniform(0.5, 1.5, N))


def _same(a, b, tol):
    assert np.array_equal(np.isinf(a), np.isinf(b)) and not np.isnan(a).any()
    f = ~np.isinf(b)
    assert np.linalg.norm(a[f] - b[f]) <= tol * np.linalg.norm(b[f])


@pytest.mark.parametrize("n", [12, 32, 33, 64])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_infinite_pivots(ct, oracle, n, prec):
    M = _matrix(n, 3, n)
    pins = [0, 3, n - 9, n + 2, M.shape[0] - 8, M.shape[0] - 1]
    A = M.copy()
    A[pins, pins] = np.inf
    A = sp.csc_matrix(A)
    P, S = ct.symbolic(A)
    print(n, prec, S.nfr, flush=True)
    tol = 1e-5 if prec == "f32" else 1e-12  # the suite's bars for the factor
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=ct.MF_FP32 if prec == "f32" else ct.MF_FP64))
    D, L, d, info = oracle.chol_impl(S, *oracle.assemble(S, P, A))
    assert info == 0 and ct.issuccess(F)
    _same(F.Dval, D, tol)
    _same(F.Lval, L, tol)


@pytest.mark.parametrize("n", [12, 32, 33, 64])
@pytest.mark.parametrize("kind", ["chol", "ldlt"])
def test_subnormal_pivots(ct, oracle, n, kind):
    """Entries around 1e-308: pivots below the normal range, reciprocals still finite."""
    M = _matrix(n, 2, n)
    A = sp.csc_matrix(M * (1.5e-308 / np.diag(M).max()))
    A.data = np.where(np.abs(A.data) < 1e-313, 0.0, A.data)
    P, S = ct.symbolic(A)
    print(n, kind, S.nfr, flush=True)
    diag = 1 if kind == "ldlt" else 0
    if diag:
        F = ct.ldlt_(ct.ChordalLDLt(A, P, S))
    else:
        F = ct.cholesky_(ct.ChordalCholesky(A, P, S))
    D, L, d, info = oracle.chol_impl(S, *oracle.assemble(S, P, A), diag=diag)
    assert info == 0 and ct.issuccess(F) and d is not None
    # entries of A are whole multiples of 2^-1074, 1.2e-15 of the smallest pivot here; a column
    # of at most 64 such roundings stays below 1e-12
    big = 2.0 ** 1000  # (norms of subnormal numbers)
    pairs = [(F.Dval, D), (F.Lval, L)] + ([(F.d, d)] if diag else [])
    for a, b in pairs:
        if b.size:
            a, b = a * big, b * big
            assert np.isfinite(a).all() and np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("n", [12, 16, 21, 32, 33, 47, 64])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_solves_with_infinite_pivots(ct, n, prec):
    """Finite solutions with a zero at every pinned unknown, column by column and in blocks."""
    M = _matrix(n, 3, n)
    pins = [0, 3, n - 9, n + 2, M.shape[0] - 8, M.shape[0] - 1]
    A = M.copy()
    A[pins, pins] = np.inf
    A = sp.csc_matrix(A)
    P, S = ct.symbolic(A)
    print(n, prec, S.nfr, flush=True)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=ct.MF_FP32 if prec == "f32" else ct.MF_FP64))
    assert ct.issuccess(F)
    free = np.setdiff1d(np.arange(M.shape[0]), pins)
    for nrhs in (1, 5, 7, 17):
        B = np.random.default_rng(nrhs).standard_normal((M.shape[0], nrhs))
        X = ct.solve(F, B)
        X0 = np.zeros_like(B)
        X0[free] = np.linalg.solve(M[np.ix_(free, free)], B[free])
        assert np.all(X[pins] == 0.0), nrhs
        # the suite's bars for solutions
        assert np.linalg.norm(X - X0) <= (1e-4 if prec == "f32" else 1e-11) * np.linalg.norm(X0), nrhs


@pytest.mark.parametrize("n", [64, 65, 100, 150, 200])
def test_given_factor_with_infinite_pivots(ct, oracle, n):
    """div_impl! on a factor from elsewhere whose big fronts have infinite diagonal entries."""
    M = _matrix(n, 3, n)
    pins = [0, 3, 40, n - 9, n + 2, M.shape[0] - 8, M.shape[0] - 1]
    A = M.copy()
    A[pins, pins] = np.inf
    P, S = ct.symbolic(sp.csc_matrix(A))
    print(n, S.nfr, flush=True)
    D, L, d, info = oracle.chol_impl(S, *oracle.assemble(S, P, sp.csc_matrix(A)))
    assert info == 0 and np.isinf(D).sum() == len(set(pins))
    perm = P.perm - 1
    free = np.setdiff1d(np.arange(M.shape[0]), pins)
    for nrhs in (1, 5, 17):
        B = np.random.default_rng(nrhs).standard_normal((M.shape[0], nrhs))
        X0 = np.zeros_like(B)
        X0[free] = np.linalg.solve(M[np.ix_(free, free)], B[free])
        X = ct.div_impl(S, D, L, None, B[perm], diag=ct.MF_CHOLESKY)
        assert np.all(X[np.isin(perm, pins)] == 0.0), nrhs
        assert np.linalg.norm(X - X0[perm]) <= 1e-11 * np.linalg.norm(X0), nrhs
