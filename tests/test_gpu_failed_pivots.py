"""GPU: failed pivots in small fronts that a workgroup factors, in the columns of each of its four
wavefronts, in the small region and above a big front.  The reported column is the oracle's, and
the fronts that do not descend from the failed one are those of the repaired matrix."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _block(rng, cols, tail, touch):
    """A dense block of `cols` columns; with `tail`, a second dense block of `tail` columns, the
    first `touch` of which couple to the first block."""
    n = cols + tail
    A = np.zeros((n, n))
    A[:cols, :cols] = rng.uniform(-1, 1, (cols, cols))
    if tail:
        A[cols:, cols:] = rng.uniform(-1, 1, (tail, tail))
        A[cols:cols + touch, :cols] = rng.uniform(-1, 1, (touch, cols))
    A = np.tril(A, -1)
    A = A + A.T
    return A + np.diag(np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n))


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("col", [0, 1, 2, 3, 4, 37, 46, 47])
@pytest.mark.parametrize("kind", ["chol", "ldlt"])
def test_failed_pivot_of_a_workgroup_front(ct, oracle, big, col, kind):
    rng = np.random.default_rng(100 * col + big)
    cols, tail, touch, count = (70, 48, 5, 6) if big else (48, 0, 0, 40)
    blocks = [_block(rng, cols, tail, touch) for _ in range(count)]
    good = sp.block_diag([sp.csc_matrix(b) for b in blocks], format="csc")
    n1 = cols + tail
    which = count // 2
    at = which * n1 + (cols + col if big else col)
    # the failing pivot: negative for Cholesky, zero for LDLt with an all-zero column beside it
    bad = good.tolil()
    if kind == "chol":
        bad[at, at] = -1e3
    else:
        s = slice(which * n1, (which + 1) * n1)
        row = np.zeros(n1)
        bad[at, s] = row
        bad[s, at] = row[:, None]
    bad = bad.tocsc()
    order = np.arange(1, good.shape[0] + 1)
    P, S = ct.symbolic(good, alg=order)
    print(big, col, kind, S.nfr, flush=True)
    diag = 1 if kind == "ldlt" else 0
    Dg, Lg, dg, ig = oracle.chol_impl(S, *oracle.assemble(S, P, good), diag=diag)
    D0, L0, d0, info0 = oracle.chol_impl(S, *oracle.assemble(S, P, bad), diag=diag)
    assert ig == 0 and info0 > 0
    for _ in range(3):
        if diag:
            F = ct.ldlt_(ct.ChordalLDLt(bad, P, S), check=False)
        else:
            F = ct.cholesky_(ct.ChordalCholesky(bad, P, S), check=False)
        assert not ct.issuccess(F) and F.info == P.perm[info0 - 1]
        lo, hi = which * n1, (which + 1) * n1
        num = den = 0.0
        for j in range(S.nfr):
            c = P.perm[S.resptr[j] - 1] - 1
            if lo <= c < hi:
                continue
            for X, Y, ptr in ((F.Dval, Dg, S.Dptr), (F.Lval, Lg, S.Lptr)):
                a = slice(ptr[j] - 1, ptr[j + 1] - 1)
                num += np.sum((X[a] - Y[a]) ** 2)
                den += np.sum(Y[a] ** 2)
        assert np.sqrt(num / den) <= 1e-12  # the suite's bar for the factor
