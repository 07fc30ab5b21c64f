"""GPU: extend-add into a big front from many children with few rows in each of its tiles, against
the oracle: fewer and more sources than are taken at a time, scattered separators (up to four, up
to eight and more columns in a wavefront's strip), windows of neighbouring rows, and mixtures
with some and with few children that cover whole tiles."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _matrix(kids, cols, ns, sep, kind, seed):
    """`kids` leaves of `cols` columns with `sep` of the `ns` separator columns each."""
    rng = np.random.default_rng(seed)
    n = kids * cols + ns
    A = np.zeros((n, n))
    for k in range(kids):
        s = slice(k * cols, (k + 1) * cols)
        A[s, s] = rng.uniform(-1, 1, (cols, cols))
        if kind == "window" or (kind == "mixed" and k % 5 == 2) or (kind == "few" and k % 50 == 7):
            m = sep if kind == "window" else min(ns, 70)
            at = rng.integers(0, ns - m + 1) + np.arange(m)
        else:
            at = rng.choice(ns, sep, replace=False)
        A[kids * cols + at, s] = rng.uniform(-1, 1, (len(at), cols))
    A[kids * cols:, kids * cols:] = rng.uniform(-1, 1, (ns, ns))
    A = np.tril(A, -1)
    A = A + A.T
    return sp.csc_matrix(A + np.diag(np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)))


CASES = [(9, 1, 150, 3, "scattered"), (70, 2, 150, 9, "scattered"), (137, 1, 200, 30, "scattered"),
         (130, 3, 65, 12, "scattered"), (200, 1, 131, 50, "scattered"), (70, 1, 150, 12, "window"),
         (66, 2, 193, 16, "window"), (70, 1, 100, 17, "window"), (90, 2, 150, 6, "mixed"), (7, 2, 150, 6, "mixed"),
         (150, 1, 150, 8, "few"), (190, 1, 70, 8, "few")]


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("kids,cols,ns,sep,kind", CASES)
@pytest.mark.parametrize("what", ["chol", "ldlt", "chol_f32"])
def test_many_children(ct, oracle, kids, cols, ns, sep, kind, what):
    A = _matrix(kids, cols, ns, sep, kind, kids + sep)
    P, S = ct.symbolic(A)
    print(what, kids, cols, ns, sep, kind, S.nfr, flush=True)
    tol = 1e-5 if what == "chol_f32" else 1e-12  # the suite's bars for the factor
    prec = ct.MF_FP32 if what == "chol_f32" else ct.MF_FP64
    diag = 1 if what == "ldlt" else 0
    D, L, d, info = oracle.chol_impl(S, *oracle.assemble(S, P, A), diag=diag)
    if diag:
        F = ct.ldlt_(ct.ChordalLDLt(A, P, S, precision=prec))
        assert _rel(F.d, d) <= tol
    else:
        F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=prec))
    assert info == 0 and ct.issuccess(F)
    assert _rel(F.Dval, D) <= tol and _rel(F.Lval, L) <= tol
