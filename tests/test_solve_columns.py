"""The planner's choice of how many right-hand sides are solved column by column (mf_plan_check,
stats[19]): none but one where tasks fill the chip, a whole block of sixteen where a chain does
not, and in between fewer with more unknowns."""
import ctypes

import numpy as np
import scipy.sparse as sp

import pytest


def _columns(ct, A, order):
    from cliquetrees_amd import _native
    P, S = ct.symbolic(A, alg=order)
    arrs = [np.ascontiguousarray(a, dtype=np.int64) for a in
            [S.resptr, S.sepptr, S.septgt, S.reltgt, S.chdptr, S.chdtgt, S.Dptr, S.Lptr]]
    st = np.zeros(20, dtype=np.int64)
    msg = ctypes.create_string_buffer(256)
    rc = _native.sym().mf_plan_check(S.n, S.nfr, *[a.ctypes.data_as(_native.i64p) for a in arrs],
                                     st.ctypes.data_as(_native.i64p), len(st), msg, 256)
    assert rc == 0, msg.value
    return int(st[19])


@pytest.mark.parametrize("what,lo,hi", [("forest", 1, 1), ("diagonal", 1, 1), ("path", 16, 16), ("dense", 16, 16),
                                        ("star", 16, 16), ("one", 1, 16)])
def test_extremes(ct, what, lo, hi):
    pr = ct.problems
    if what == "forest":
        A, order = sp.block_diag([pr.grid_laplacian_random((5 + i % 4, 6), i) for i in range(2000)], format="csc"), "mmd"
    elif what == "diagonal":
        A, order = sp.csc_matrix(2.0 * sp.eye(100000)), None
    elif what == "path":
        A, order = sp.csc_matrix(sp.diags([-np.ones(9999), np.full(10000, 3.0), -np.ones(9999)], [-1, 0, 1])), "mmd"
    elif what == "dense":
        A, order = sp.csc_matrix(np.ones((300, 300)) + 300 * np.eye(300)), None
    elif what == "star":
        B = sp.csc_matrix(np.ones((20, 4000)))
        A, order = sp.bmat([[4000.0 * sp.eye(4000), B.T], [B, 1e5 * sp.eye(20)]], format="csc"), None
    else:
        A, order = sp.csc_matrix([[2.0]]), None
    A.sort_indices()
    assert lo <= _columns(ct, A, order) <= hi


def test_fewer_columns_with_more_unknowns(ct):
    pr = ct.problems
    c = [_columns(ct, pr.laplacian3d_7pt(m, m, m, 0), ct.grid_nd(m, m, m)) for m in (12, 20, 32, 48)]
    assert c[0] == 16 and all(a >= b for a, b in zip(c, c[1:])) and 3 <= c[-1] <= 7
