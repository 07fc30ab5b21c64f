"""GPU: the tile products and gathers of the selected inversion at the edges of their 32- and
64-wide tiles, against the dense inverse.

Two dense blocks coupled to a dense separator set the sizes of a front's columns, of its update
rows and of the root directly; a third level comes from a chain of separators."""
import numpy as np
import pytest
import scipy.sparse as sp

from densehelp import dense_lower, permuted_dense

pytestmark = pytest.mark.gpu

# (block, separator): small fronts, one tile of each kind, one column past 32, 64, 96 and 128,
# update rows past one and several tiles
SIZES = [(20, 30), (31, 34), (33, 33), (65, 1), (64, 64), (96, 97), (97, 65), (33, 129), (129, 127), (200, 150)]


def _matrix(sizes, seed):
    """Blocks of the given sizes; block 0 and 1 couple to block 2, block k to block k + 1 after that."""
    rng = np.random.default_rng(seed)
    at = np.concatenate([[0], np.cumsum(sizes)])
    n = at[-1]
    A = np.zeros((n, n))
    for k in range(len(sizes)):
        up = max(k + 1, 2)
        for j in {k, up} - {len(sizes)}:
            A[at[j]:at[j + 1], at[k]:at[k + 1]] = rng.uniform(-1, 1, (sizes[j], sizes[k]))
    A = np.tril(A, -1)
    A = A + A.T
    return sp.csc_matrix(A + np.diag(np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)))


@pytest.mark.parametrize("nb,ns", SIZES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tile_edges(ct, nb, ns, precision):
    A = _matrix([nb, nb, ns, ns // 2 + 1, 70], nb + ns)
    P, S = ct.symbolic(A)
    print(nb, ns, precision, S.nfr, flush=True)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=ct.MF_FP32 if precision == "fp32" else ct.MF_FP64))
    ct.selinv_(F)
    got = dense_lower(S, F.Dval, F.Lval)
    on = dense_lower(S, np.ones(S.ndz), np.ones(S.nlz)) != 0
    want = np.where(on, np.linalg.inv(permuted_dense(A, P)), 0.0)
    # diagonally dominant: n eps with the margin of the tile tests
    tol = 1e-4 if precision == "fp32" else 1e-12
    assert np.linalg.norm(np.where(on, got, 0.0) - want) <= tol * np.linalg.norm(want)
