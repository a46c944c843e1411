"""The LU panel's kernels (leaf factorisation with its columns in registers, row
interchanges, triangular-solve leaf) at the sizes where their forms change: leaves
of up to 512, 1024, 2048, 4096 and more rows, and one row either side."""
import ctypes as C
import os

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe():
    import qbhip
    return C.CDLL(os.path.join(HERE, "native", "libqbt_linalg.so")), C.c_void_p(
        qbhip.default_context().ptr.value)


def _p(a):
    return C.c_void_p(a.ctypes.data)


def _getrf(probe, A):
    """A: (batch, n, n) with A[b][column][row]; returns the factors and pivots."""
    L, ctx = probe
    b, n, _ = A.shape
    F, ipiv = np.ascontiguousarray(A), np.zeros((b, n), np.int32)
    f = L.qbt_getrf_c128 if A.dtype == np.complex128 else L.qbt_getrf_c64
    assert f(ctx, n, _p(F), _p(ipiv), b) == 0
    return F, ipiv


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 31, 33, 255, 257, 512, 513, 1024, 1025, 2048, 2049, 4097])
def test_known_factors(probe, n, dt):
    """A = P^T L U with sparse dyadic factors: every step's pivot is unique
    (|re| + |im| of L below 1) and every sum is exact in the operand type, so
    the pivots are known, and within one panel (n <= 256) the factors are the
    given ones bit for bit.  Between panels a trailing update may round: there
    the factors are held to 64 u times the largest entry."""
    rng = np.random.default_rng(n)
    units = np.array([1, -1, 1j, -1j])

    def tri(scale, lower):
        k = 5 * n
        i, j = rng.integers(0, n, k), rng.integers(0, n, k)
        ok = i > j if lower else i < j
        v = rng.choice(scale, k) * rng.choice(units, k)
        M = sp.coo_matrix((v[ok], (i[ok], j[ok])), shape=(n, n)).tocsr()
        M.data = np.where(np.abs(M.data) > 0.5, 0.5, M.data) if lower else M.data
        return M

    Lm = tri([0.5, 0.25], True) + sp.identity(n, dtype=complex)
    Um = tri([1.0, 2.0], False) + sp.diags(rng.choice([4.0, 8.0], n) * rng.choice(units, n))
    perm = rng.permutation(n)
    A = np.empty((n, n), complex)
    A[perm] = (Lm @ Um).toarray()  # row perm[i] of A is row i of L U
    F, ipiv = _getrf(probe, np.ascontiguousarray(A.T[None]).astype(dt))
    order = np.arange(n)
    for s, q in enumerate(ipiv[0]):
        order[s], order[q] = order[q], order[s]
    assert np.array_equal(order, perm)
    ref = (sp.tril(Lm, -1) + Um).toarray()
    if n <= 256:
        assert np.array_equal(F[0].T, ref.astype(dt))
    else:
        u = np.finfo(dt).eps / 2
        assert np.max(np.abs(F[0].T - ref)) <= 64 * u * np.max(np.abs(ref))


@pytest.mark.parametrize("dt", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [20, 300, 700, 1500])
def test_ties_zero_columns_and_nan(probe, n, dt):
    """Of equal candidates the first row is the pivot; a column without a
    nonzero entry stays unscaled (lu!(check=false)); a NaN is never chosen."""
    rng = np.random.default_rng(n)
    A = np.zeros((3, n, n), dt)
    A[0, 0] = 1  # a column of equal entries: no interchange
    A[0, 0, n // 2:] = -1j
    idx = np.arange(n)
    A[0, idx[1:], idx[1:]] = 2
    A[1, idx, idx] = 1  # identity but for a zero column
    A[1, 3, 3] = 0
    A[2] = (rng.standard_normal((n, n)) * 0.1).astype(dt)
    A[2, idx, idx] = 3
    A[2, 0, 5] = np.nan
    A[2, 0, 9] = 7
    F, ipiv = _getrf(probe, A)
    assert ipiv[0, 0] == 0
    assert np.allclose(F[0, 0, 1:], A[0, 0, 1:]) and F[0, 0, 0] == 1
    assert np.array_equal(ipiv[1], idx) and np.array_equal(F[1], A[1])
    assert ipiv[2, 0] == 9 and F[2, 0, 0] == 7
