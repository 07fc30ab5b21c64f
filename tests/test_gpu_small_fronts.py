"""GPU: the small-front kernels (one wavefront up to nJ = 32, one workgroup up to 64) at the
sizes where they can go wrong, against the oracle: groups of four columns, the last column, no
update rows, one child and more children than are taken at a time, and a failed pivot."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

# (children, their columns, separator): children of nn = columns, na = separator under one root
SHAPES = [(1, 1, 1), (2, 1, 31), (2, 3, 29), (3, 4, 28), (2, 5, 28), (5, 16, 16), (2, 31, 1), (70, 2, 20),
          (2, 1, 63), (3, 7, 57), (2, 8, 56), (4, 33, 31), (2, 60, 4), (2, 63, 1), (70, 3, 50), (1, 64, 64)]


def _matrix(kids, cols, ns, seed, indefinite):
    rng = np.random.default_rng(seed)
    n = kids * cols + ns
    A = np.zeros((n, n))
    for k in range(kids):
        s = slice(k * cols, (k + 1) * cols)
        A[s, s] = rng.uniform(-1, 1, (cols, cols))
    A[kids * cols:, :] = rng.uniform(-1, 1, (ns, n))
    A = np.tril(A, -1)
    A = A + A.T
    d = np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)  # diagonally dominant: every factor exists
    if indefinite:
        d *= np.where(rng.random(n) < 0.3, -1.0, 1.0)
    return sp.csc_matrix(A + np.diag(d))


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("kids,cols,ns", SHAPES)
@pytest.mark.parametrize("kind", ["chol", "ldlt", "chol_f32"])
def test_small_fronts(ct, oracle, kids, cols, ns, kind):
    A = _matrix(kids, cols, ns, 10 * cols + ns, kind == "ldlt")
    P, S = ct.symbolic(A)
    print(kind, kids, cols, ns, S.nfr, flush=True)
    Dv, Lv = oracle.assemble(S, P, A)
    prec = ct.MF_FP32 if kind == "chol_f32" else ct.MF_FP64
    # the suite's bars for the factor
    tol = 1e-5 if kind == "chol_f32" else 1e-12
    if kind == "ldlt":
        F = ct.ldlt_(ct.ChordalLDLt(A, P, S, precision=prec))
        D, L, d, info = oracle.chol_impl(S, Dv, Lv, diag=1)
        assert _rel(F.d, d) <= tol
    else:
        F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=prec))
        D, L, d, info = oracle.chol_impl(S, Dv, Lv)
    assert info == 0 and ct.issuccess(F)
    assert _rel(F.Dval, D) <= tol
    assert L.size == 0 or _rel(F.Lval, L) <= tol


@pytest.mark.parametrize("kids,cols,ns,bad", [(2, 3, 20, 4), (3, 8, 40, 13), (2, 5, 20, 25)])
def test_failed_pivot(ct, oracle, kids, cols, ns, bad):
    """The first column of a failed pivot, as the oracle reports it."""
    A = _matrix(kids, cols, ns, 5, False).tolil()
    A[bad, bad] = -50.0
    A = A.tocsc()
    P, S = ct.symbolic(A)
    Dv, Lv = oracle.assemble(S, P, A)
    D, L, d, info = oracle.chol_impl(S, Dv, Lv)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S), check=False)
    assert info > 0 and not ct.issuccess(F) and F.info == P.perm[info - 1]
