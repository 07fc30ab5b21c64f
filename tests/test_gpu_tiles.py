"""GPU: the dense tile kernels of big fronts at the sizes where they can go wrong (edges of the
16-column blocks and of the 64- and 128-wide tiles), against the oracle.

A matrix of two dense blocks coupled to a dense separator has three fronts: the blocks' fronts
(nn = block size, na = separator size) and the separator's (nn = its size, na = 0), so the sizes
of the panel, of its update rows and of the root are set directly."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

# (block, separator): 16-column blocks of the diagonal tile, one column past them, tiles of one
# and two panel columns with ragged last tiles, wide update-matrix tiles (block >= 128) with
# remainders, long trailing updates (more than eight panel steps)
SIZES = [(65, 1), (79, 17), (80, 64), (81, 65), (127, 63), (128, 128), (129, 129), (143, 191), (193, 66),
         (257, 130), (700, 75), (64, 641)]


def _matrix(nb, ns, seed, indefinite):
    rng = np.random.default_rng(seed)
    n = 2 * nb + ns
    A = np.zeros((n, n))
    for k, m in ((0, nb), (nb, nb), (2 * nb, ns)):
        A[k:k + m, k:k + m] = rng.uniform(-1, 1, (m, m))
    A[2 * nb:, :2 * nb] = rng.uniform(-1, 1, (ns, 2 * nb))
    A = np.tril(A, -1)
    A = A + A.T
    d = np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)  # diagonally dominant: every factor exists
    if indefinite:
        d *= np.where(rng.random(n) < 0.3, -1.0, 1.0)
    return sp.csc_matrix(A + np.diag(d)), np.sign(d)


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("nb,ns", SIZES)
@pytest.mark.parametrize("kind", ["chol", "ldlt", "ldlt_signs", "chol_f32"])
def test_tile_edges(ct, oracle, nb, ns, kind):
    ldlt, f32 = kind.startswith("ldlt"), kind.endswith("f32")
    A, signs = _matrix(nb, ns, 1000 * nb + ns, ldlt)
    P, S = ct.symbolic(A)
    print(kind, nb, ns, S.nfr, flush=True)
    Dv, Lv = oracle.assemble(S, P, A)
    prec = ct.MF_FP32 if f32 else ct.MF_FP64
    if ldlt:
        F = ct.ldlt_(ct.ChordalLDLt(A, P, S, precision=prec), signs=signs if kind == "ldlt_signs" else None)
        D, L, d, info = oracle.chol_impl(S, Dv, Lv, diag=1)
    else:
        F = ct.cholesky_(ct.ChordalCholesky(A, P, S, precision=prec))
        D, L, d, info = oracle.chol_impl(S, Dv, Lv)
    assert info == 0 and ct.issuccess(F)
    # the suite's bars for the factor (1e-12 in FP64, 1e-5 in FP32); residual of a diagonally
    # dominant system: n eps (1.6e-13, 9e-5)
    tol, rtol = (1e-5, 1e-4) if f32 else (1e-12, 1e-12)
    assert _rel(F.Dval, D) <= tol and _rel(F.Lval, L) <= tol
    if ldlt:
        assert _rel(F.d, d) <= tol
    B = np.random.default_rng(5).standard_normal((A.shape[0], 3))
    X = ct.solve(F, B)
    assert np.linalg.norm(A @ X - B) <= rtol * np.linalg.norm(B)


@pytest.mark.parametrize("kids,rows,ns", [(80, 20, 150), (70, 150, 150), (3, 65, 129), (130, 5, 66)])
def test_extend_add_many_children(ct, oracle, kids, rows, ns):
    """A root front whose tiles take from one child up to more children than a wavefront has
    lanes, with scattered and with complete row sets."""
    rng = np.random.default_rng(kids + rows)
    nb = 3
    n = nb * kids + ns
    A = np.zeros((n, n))
    for k in range(kids):
        r = np.sort(rng.choice(ns, size=min(rows, ns), replace=False)) + nb * kids
        A[np.ix_(r, range(nb * k, nb * k + nb))] = rng.uniform(-1, 1, (len(r), nb))
        A[nb * k:nb * k + nb, nb * k:nb * k + nb] = rng.uniform(-1, 1, (nb, nb))
    A[nb * kids:, nb * kids:] = rng.uniform(-1, 1, (ns, ns))
    A = np.tril(A, -1)
    A = A + A.T
    A = sp.csc_matrix(A + np.diag(np.abs(A).sum(1) + 1.0))
    P, S = ct.symbolic(A)
    print(kids, rows, ns, S.nfr, flush=True)
    Dv, Lv = oracle.assemble(S, P, A)
    D, L, d, info = oracle.chol_impl(S, Dv, Lv)
    F = ct.cholesky_(ct.ChordalCholesky(A, P, S))
    assert info == 0 and _rel(F.Dval, D) <= 1e-12 and _rel(F.Lval, L) <= 1e-12


@pytest.mark.parametrize("sizes", [[65], [150], [700], [1500], [200] * 12])
@pytest.mark.parametrize("wg_per_cu", [0, 1])
@pytest.mark.parametrize("kind", ["chol", "ldlt", "chol_f32"])
def test_diagonal_chain(ct, sizes, wg_per_cu, kind):
    """Chains of two to twenty-four diagonal tiles, one of them or several at once: a workgroup
    goes on to the next tile where its ticket has been handed out (short lists, all at once) and
    leaves it to the ticket's holder where it has not (long lists, fewer workgroups)."""
    rng = np.random.default_rng(len(sizes) + sizes[0])
    n = sum(sizes)
    A = np.zeros((n, n))
    at = 0
    for m in sizes:
        A[at:at + m, at:at + m] = rng.uniform(-1, 1, (m, m))
        at += m
    A = np.tril(A, -1)
    A = A + A.T
    d = np.abs(A).sum(1) + rng.uniform(0.5, 1.5, n)
    if kind == "ldlt":
        d *= np.where(rng.random(n) < 0.3, -1.0, 1.0)
    A += np.diag(d)
    C = sp.csc_matrix(A)
    P, S = ct.symbolic(C)
    print(kind, sizes, wg_per_cu, S.nfr, flush=True)
    prec = ct.MF_FP32 if kind == "chol_f32" else ct.MF_FP64
    tuning = [0, 0, 0, 0, 0, 0, 1, wg_per_cu]  # 0: the default
    make = ct.ChordalLDLt if kind == "ldlt" else ct.ChordalCholesky
    F = make(C, P, S, precision=prec, tuning=tuning)
    F = ct.ldlt_(F) if kind == "ldlt" else ct.cholesky_(F)
    assert ct.issuccess(F)
    B = rng.standard_normal((n, 2))
    X = ct.solve(F, B)
    # diagonally dominant: n eps with the margin of the other tile tests
    assert np.linalg.norm(A @ X - B) <= (1e-4 if kind == "chol_f32" else 1e-12) * np.linalg.norm(B)
