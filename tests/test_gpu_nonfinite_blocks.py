"""GPU: infinities and NaN in right-hand sides of the blocked solves (blocks of sixteen columns):
every wait ends, and the other columns of the block and of the other blocks stay as they were."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["big", "forest"])
def test_nonfinite_columns_of_a_block(ct, what):
    if what == "big":
        A, order = ct.problems.grid_laplacian_random((90, 80), 1), ct.grid_nd(90, 80, 1)
    else:
        A, order = sp.block_diag([ct.problems.grid_laplacian_random((5, 4 + i % 3), i) for i in range(300)] * 4,
                                 format="csc"), "mmd"
    P, S = ct.symbolic(A, alg=order)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S))
    n, cols = A.shape[0], 37
    B = np.random.default_rng(1).standard_normal((n, cols))
    good = ct.solve(F, B)
    odd = np.array([np.nan, np.inf, 0.0, 0.0])
    # signalling NaNs of both halves of the payload range
    odd[2:] = np.array([0x7FF4A5A5DEADBEE1, 0x7FF0000000000001], dtype=np.uint64).view(np.float64)
    for v in odd:
        for row, col in ((0, 0), (n // 2, 17), (n - 1, 36), (n // 3, 15)):
            print(what, v, row, col, flush=True)
            D = B.copy()
            D[row, col] = v
            X = ct.solve(F, D)
            rest = np.arange(cols) != col
            assert not np.isfinite(X[:, col]).all()
            assert np.array_equal(X[:, rest], good[:, rest])
