"""GPU: GMW81 on one dense front whose block columns have 1023 to 0, 1024 to 0 and 1025 to 1 rows
below the diagonal tile: the heights at which the diagonal task changes how many rows and columns
it reads at a time (256, 512, 1024), against the oracle."""
import numpy as np
import pytest
import scipy.sparse as sp

from densehelp import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1087, 1088, 1089])
@pytest.mark.parametrize("diag", [0, 1])
def test_heights(ct, oracle, n, diag):
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n))
    A = np.tril(A, -1)
    A = A + A.T
    d = np.abs(A).sum(1)
    d[rng.random(n) < 0.1] *= -0.5  # pivots that the rule has to change
    A = sp.csc_matrix(A + np.diag(d))
    P, S = ct.symbolic(A)
    print(n, diag, S.nfr, flush=True)
    signs = np.ones(n) if diag else None
    sg = None if signs is None else np.ascontiguousarray(signs[P.perm - 1])
    D0, L0, d0, info = oracle.chol_impl(S, *oracle.assemble(S, P, A), diag, signs=sg, reg=("gmw81", -1.0, -1.0))
    assert info == 0
    if diag:
        F = ct.ChordalLDLt(A, P, S)
        ct.ldlt_(F, signs=signs, reg=ct.GMW81())
        assert rel(F.d, d0) <= 1e-12  # the suite's bar
    else:
        F = ct.ChordalCholesky(A, P, S)
        ct.cholesky_(F, reg=ct.GMW81())
    assert ct.issuccess(F) and rel(F.Dval, D0) <= 1e-12
