"""GPU: the explicit zeros of the internal fronts stay within the fraction a caller asks for, at
every front size; the default rule and its value read back give the same plan."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fronts(ct, S, tuning):
    from cliquetrees_amd import _native
    lib = _native.hip()
    pl = ct.device_plan(S, tuning)
    st = np.zeros(3, np.int64)
    lib.mf_plan_stats(pl.handle, st.ctypes.data_as(_native.i64p), 3)
    out = np.zeros((int(st[2]), 5), np.int64)
    assert lib.mf_plan_fronts(pl.handle, out.ctypes.data_as(_native.i64p), out.size) >= 0
    return pl, out


@pytest.mark.parametrize("ppm", [1, 5000, 20000, 100000])
@pytest.mark.parametrize("grid", ["plane", "box"])
def test_zero_fraction(ct, ppm, grid):
    if grid == "plane":
        A, order = ct.problems.grid_laplacian_random((70, 60), 0), "mmd"
    else:
        A, order = ct.problems.laplacian3d_7pt(14, 15, 13, seed=1), ct.grid_nd(14, 15, 13)
    P, S = ct.symbolic(A, alg=order)
    # entries of every column of the factor
    count = np.zeros(S.n, np.int64)
    for j in range(S.nfr):
        nn, na = int(S.nn()[j]), int(S.na()[j])
        count[S.resptr[j] - 1:S.resptr[j + 1] - 1] = np.arange(nn, 0, -1) + na
    _, fr = _fronts(ct, S, [0, 0, 0, 0, ppm, -1, -1, -1])
    for c0, nn, na, parent, small in fr:
        size = nn * (nn + 1) // 2 + nn * na
        zeros = size - int(count[c0:c0 + nn].sum())
        # (a panel of at most eight columns is merged whatever it holds)
        assert zeros >= 0 and (nn <= 8 or zeros <= 1e-6 * ppm * size), (c0, nn, na, zeros / size)
    base, f0 = _fronts(ct, S, None)
    back = base.tuning()
    assert back["zero_ppm"] == 50000
    _, f1 = _fronts(ct, S, [back[k] for k in ("upd_group", "ea_rows", "wide_k", "sim_workers", "zero_ppm", "prio", "fuse",
                                              "wg_per_cu")])
    assert np.array_equal(f0, f1)
