"""The complex128 product on the int8 matrix cores (qb_rns.hip) against products in
extended precision, at the edges of its tiles and of its operands' range."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
U = 2.0 ** -53


@pytest.fixture(scope="module")
def probe():
    import qbhip
    return C.CDLL(os.path.join(HERE, "native", "libqbt_rns.so")), C.c_void_p(
        qbhip.default_context().ptr.value)


def _p(a):
    return C.c_void_p(a.ctypes.data)


def _sub(probe, A, B, Cm):
    """Cm - A B per matrix; arrays [batch][column][row] (column-major matrices)."""
    L, ctx = probe
    b, K, M = A.shape
    N = B.shape[1]
    out = np.array(Cm, order="C")  # the product updates it in place
    t = (C.c_double * 2)()
    rc = L.qbt_rns_sub(ctx, M, N, K, _p(np.ascontiguousarray(A)), _p(np.ascontiguousarray(B)),
                       _p(out), b, 0, C.byref(t, 0), C.byref(t, 8))
    assert rc == 0
    return out


def _rand(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


# one tile, edges one below and above the 128 x 64 tile and the 32 x 32 wave tiles,
# several 512 x 512 groups of tiles and several matrices
@pytest.mark.parametrize("M,N,K,b", [(1, 1, 512, 1), (31, 33, 512, 2), (127, 65, 512, 1),
                                     (128, 64, 512, 1), (129, 63, 512, 3), (530, 517, 512, 2),
                                     (300, 1100, 512, 2)])
@pytest.mark.parametrize("spread", [0.0, 300.0])
def test_product(probe, M, N, K, b, spread):
    """Operands rounded at 2^-53 of their row's / column's largest component and
    an exact product: |error| <= 4 u sqrt(2 K) max_k|a_ik| ||b_j|| + u-sized roundings
    of the product and of C (u = 2^-53).  spread: rows and columns scaled by powers
    of two up to 2^+-spread."""
    rng = np.random.default_rng(M * 7 + N)
    A, B, C0 = _rand(rng, (b, K, M)), _rand(rng, (b, N, K)), _rand(rng, (b, N, M))
    if spread:
        A *= 2.0 ** rng.integers(-spread, spread, (b, 1, M))
        B *= 2.0 ** rng.integers(-spread, spread, (b, N, 1))
        C0 *= 0
    R = _sub(probe, A, B, C0)
    for i in range(b):
        a, w, c = (x.T.astype(np.clongdouble) for x in (A[i], B[i], C0[i]))
        ref = c - a @ w if M * N * K < 3e7 else (C0[i].T - A[i].T @ B[i].T)
        mag = np.sqrt(2.0 * K) * (np.max(np.abs(A[i]), 0)[:, None] * np.linalg.norm(B[i], axis=1)
                                  + np.linalg.norm(A[i], axis=0)[:, None] * np.max(np.abs(B[i]), 1))
        tol = 4 * U * (mag + np.abs(C0[i].T))
        assert np.all(np.abs(R[i].T - ref) <= tol)


def test_exact_zero_and_nonfinite(probe):
    """Small integers give the exact product up to one rounding; zero rows and
    columns leave C as it is; an infinity or NaN in a row of A or a column of B
    makes that row or column of the result NaN and no other; denormal operands
    do not disturb their neighbours."""
    rng = np.random.default_rng(3)
    M, N, K = 70, 50, 512
    A = (rng.integers(-9, 10, (1, K, M)) + 1j * rng.integers(-9, 10, (1, K, M)))
    B = (rng.integers(-9, 10, (1, N, K)) + 1j * rng.integers(-9, 10, (1, N, K)))
    C0 = _rand(rng, (1, N, M))
    A[0, :, 5] = 0
    B[0, 7] = 0
    R = _sub(probe, A, B, np.zeros_like(C0))
    exact = A[0].T @ B[0].T
    assert np.max(np.abs(R[0].T + exact)) <= 4 * U * np.max(np.abs(exact))
    R = _sub(probe, A, B, C0)
    assert np.array_equal(R[0, :, 5], C0[0, :, 5]) and np.array_equal(R[0, 7], C0[0, 7])
    A[0, 100, 9] = np.inf
    B[0, 11, 3] = np.nan
    A[0, :, 20] = 5e-324
    R2 = _sub(probe, A, B, C0)
    bad = np.zeros((N, M), bool)
    bad[:, 9] = True
    bad[11] = True
    assert np.all(np.isnan(R2[0][bad]))
    bad[:, 20] = True
    assert np.array_equal(R2[0][~bad], R[0][~bad])
    assert np.allclose(np.delete(R2[0, :, 20], 11), np.delete(C0[0, :, 20], 11), rtol=0, atol=1e-300)


@pytest.mark.parametrize("n", [4096, 4609])
def test_factors_with_and_without_residue_buffers(probe, n):
    """An LU backward error of at most 8 n u |L||U| (row sums against a vector)
    either way, the same pivots for well separated ones, and no buffer left."""
    import qbhip
    ctx = qbhip.default_context()
    L = C.CDLL(os.path.join(HERE, "native", "libqbt_linalg.so"))
    rng = np.random.default_rng(n)
    A = _rand(rng, (2, n, n))
    A[:, np.arange(n), (np.arange(n) * 7) % n] += 200.0  # the pivot of every column
    x = _rand(rng, n)
    piv = []
    try:
        for on in (True, False):
            ctx.set_residue_buffers(on)
            F, ipiv = A.copy(), np.zeros((2, n), np.int32)
            assert L.qbt_getrf_c128(C.c_void_p(ctx.ptr.value), n, _p(F), _p(ipiv), 2) == 0
            piv.append(ipiv)
            for i in range(2):
                M, order = F[i].T, np.arange(n)
                for s, q in enumerate(ipiv[i]):
                    order[s], order[q] = order[q], order[s]
                Lf, Uf = np.tril(M, -1), np.triu(M)
                y = Uf @ x
                err = np.max(np.abs(A[i].T[order] @ x - (Lf @ y + y)))
                ay = np.abs(Uf) @ np.abs(x)
                assert err <= 8 * n * U * np.max(np.abs(Lf) @ ay + ay)
    finally:
        ctx.set_residue_buffers(True)
    assert np.array_equal(piv[0], piv[1])


def test_footprint_without_residues():
    """The footprint counts what the LU takes beyond the solve buffers, for FP64
    windows of 4096 rows and more."""
    from qbhip.beyn import footprint
    for N, nq, prec, r in [(4096, 32, "fp64", 64), (8192, 48, "fp64", 64)]:
        assert footprint(N, nq, prec, r) > footprint(N, nq, prec, r, residues=False)
    for N, nq, prec, r in [(4096, 32, "fp64", 1024), (4095, 32, "fp64", 64),
                           (8192, 48, "mixed", 64)]:
        assert footprint(N, nq, prec, r) == footprint(N, nq, prec, r, residues=False)
