"""GPU: solves of 1 to 17 right-hand sides with plans that take all, some and none of them column by
column, against LAPACK, and the solve without allocation in the same forms."""
import ctypes

import numpy as np
import pytest
import scipy.linalg
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _system(ct, what):
    pr = ct.problems
    if what == "forest":  # one column
        return sp.block_diag([pr.grid_laplacian_random((5 + i % 4, 6), i) for i in range(60)] * 8, format="csc"), "mmd"
    if what == "plane":  # a few
        return pr.grid_laplacian_random((50, 45), 1), ct.grid_nd(50, 45, 1)
    if what == "box":  # most
        return pr.laplacian3d_7pt(11, 12, 13, seed=2), ct.grid_nd(11, 12, 13)
    rng = np.random.default_rng(3)
    B = sp.csc_matrix(rng.uniform(-1, 1, (70, 900)) * (rng.random((70, 900)) < 0.2))
    return sp.csc_matrix(sp.bmat([[40.0 * sp.eye(900), B.T], [B, 400.0 * sp.eye(70)]])), None  # a star


@pytest.mark.parametrize("what", ["forest", "plane", "box", "star"])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_columns(ct, what, prec):
    import torch
    from cliquetrees_amd import _native
    A, order = _system(ct, what)
    A = sp.csc_matrix(A)
    A.sort_indices()
    n = A.shape[0]
    P, S = ct.symbolic(A, alg=order)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=ct.MF_FP32 if prec == "f32" else ct.MF_FP64))
    lu = scipy.linalg.cho_factor(A.toarray(), lower=True) if n < 4000 else None
    solve = (lambda b: scipy.linalg.cho_solve(lu, b)) if lu else sp.linalg.splu(A).solve
    tol = 1e-4 if prec == "f32" else 1e-11  # the suite's bars for solutions
    perm = np.ascontiguousarray(P.perm, dtype=np.int64)
    for nrhs in (1, 2, 3, 5, 6, 9, 15, 16, 17):
        print(what, prec, n, nrhs, flush=True)
        B = np.random.default_rng(nrhs).standard_normal((n, nrhs))
        X0 = solve(B)
        X = ct.solve(F, B)
        assert np.linalg.norm(X - X0) <= tol * np.linalg.norm(X0)
        T = torch.tensor(np.ascontiguousarray(B.T), device="cuda")
        torch.cuda.synchronize()
        assert _native.hip().mf_solve_noalloc(F._f.handle, perm.ctypes.data_as(_native.i64p),
                                              ctypes.c_void_p(T.data_ptr()), nrhs, n) == 0
        assert _native.hip().mf_factor_sync(F._f.handle) == 0
        assert np.linalg.norm(T.cpu().numpy().T - X0) <= tol * np.linalg.norm(X0)


@pytest.mark.parametrize("k,m", [(9000, 2), (2500, 40)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_groups_of_blocks(ct, k, m, prec):
    """Many small systems: one to four blocks of columns to a ticket, the last one short."""
    rng = np.random.default_rng(m)
    L = np.tril(rng.uniform(-1, 1, (k, m, m)), -1)
    M = L + L.transpose(0, 2, 1)
    M[:, np.arange(m), np.arange(m)] = np.abs(M).sum(2) + rng.uniform(0.5, 1.5, (k, m))
    i = np.arange(k)[:, None, None] * m + np.arange(m)[None, :, None] + np.zeros((1, 1, m), int)
    A = sp.csc_matrix((M.ravel(), (i.ravel(), i.transpose(0, 2, 1).ravel())), shape=(k * m, k * m))
    A.sort_indices()
    P, S = ct.symbolic(A)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=ct.MF_FP32 if prec == "f32" else ct.MF_FP64))
    for nrhs in (17, 50, 70):
        print(k, m, prec, nrhs, flush=True)
        B = rng.standard_normal((k * m, nrhs))
        X0 = np.linalg.solve(M, B.reshape(k, m, nrhs)).reshape(k * m, nrhs)
        X = ct.solve(F, B)
        assert np.linalg.norm(X - X0) <= (1e-4 if prec == "f32" else 1e-11) * np.linalg.norm(X0)
