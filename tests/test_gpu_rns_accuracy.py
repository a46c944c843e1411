"""How far the residue product (qb_rns.hip) is off: its bound by row and column maxima,
also for operands graded along k, and its error on LU factors of the library's own
matrices against that of the FP64 tiles."""
import ctypes as C
import os

import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
U = 2.0 ** -53
K = 512


@pytest.fixture(scope="module")
def product():
    """-A B by the residues (rns=True) or the FP64 tiles; A: (M, 512), B: (512, N)."""
    import qbhip
    ctx = C.c_void_p(qbhip.default_context().ptr.value)
    rns = C.CDLL(os.path.join(HERE, "native", "libqbt_rns.so"))
    lin = C.CDLL(os.path.join(HERE, "native", "libqbt_linalg.so"))

    def f(A, B, use_rns):
        M, N = A.shape[0], B.shape[1]
        a, b, c = A.T.copy(order="C"), B.T.copy(order="C"), np.zeros((N, M), complex)
        p = [C.c_void_p(x.ctypes.data) for x in (a, b, c)]
        t = (C.c_double * 2)()
        rc = (rns.qbt_rns_sub(ctx, M, N, K, *p, 1, 0, C.byref(t, 0), C.byref(t, 8)) if use_rns
              else lin.qbt_gemm_sub_c128(ctx, M, N, K, *p, 1))
        assert rc == 0
        return c.T
    return f


def _exact(A, B):
    return -(A.astype(np.clongdouble) @ B.astype(np.clongdouble))


def _comp(x):
    return np.maximum(np.abs(x.real), np.abs(x.imag))


@pytest.mark.parametrize("grading", [0, 10, 20, 40])
def test_bound_with_operands_graded_along_k(product, grading):
    """Entries of A fall by 2^-grading along k and those of B grow by as much.  Operands
    within u of their row's / column's largest component per component (2 u of it, as a
    modulus, with room), fraction words that err by at most 16 moduli x 242 x 2^-73 of
    2^117.7, that is 13 u of the product of the maxima, and the result's rounding."""
    rng = np.random.default_rng(grading)
    M, N = 150, 130
    g = np.exp2(-np.floor(np.linspace(0, grading, K)))
    A = (rng.standard_normal((M, K)) + 1j * rng.standard_normal((M, K))) * g
    B = (rng.standard_normal((K, N)) + 1j * rng.standard_normal((K, N))) / g[:, None]
    R, ref = product(A, B, True), _exact(A, B)
    m, n = _comp(A).max(1)[:, None], _comp(B).max(0)[None, :]
    tol = (2 * U * (m * np.abs(B).sum(0)[None, :] + n * np.abs(A).sum(1)[:, None])
           + 16 * U * m * n + 2 * U * np.abs(ref))
    assert np.all(np.abs(R - ref) <= tol)


@pytest.mark.parametrize("op,shape,N,k", [("cfie", "star", 1100, 90 + 0.5j), ("cfie", "star", 1100, 90 - 0.5j),
                                          ("cfie", "hole", 1150, 85 + 0.35j), ("dlp", "ellipse", 1101, 130 - 0.3j),
                                          ("cfie", "ellipse", 1100, 130.25 + 0j)])
def test_no_further_off_than_the_fp64_tiles_on_factors(product, op, shape, N, k):
    """The first trailing update of the LU of T(k): largest and mean error of the residue
    product, relative to |L||U|, against those of the FP64 tile that it replaces."""
    import qbhip as q
    b = {"star": lambda: q.make_star_polar_boundary(1.0, 0.2, 5), "ellipse": lambda: q.make_full_ellipse(1.0, 0.6),
         "hole": lambda: q.CircularHoleBilliard(1.0, holes=[(0.3, 0.35, 0.0)])}[shape]()
    solver = (q.DLP_kress if op == "dlp" else q.CFIE_kress)(10.0, b)
    Ns = [N - N // 4, N // 4] if shape == "hole" else [N]
    pts = q.evaluate_points(solver, b, k.real, N=Ns)
    lu, _ = sla.lu_factor(q.assemble(solver, pts, [k], n_panels_h=9000, M_h=9, n_panels_j=4000, M_j=9)[0])
    A, B = lu[K:K + 200, :K], lu[:K, K:K + 190]
    ref, size = _exact(A, B), np.abs(A) @ np.abs(B)
    e = [np.abs(product(A, B, r) - ref) / size for r in (True, False)]
    assert e[0].max() <= e[1].max() and e[0].mean() <= e[1].mean()
