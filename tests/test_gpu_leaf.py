"""The LU panel's leaf and the triangular-solve leaf: a term rounds the running value once,
after its product, and the solves at the edges of their sizes."""
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


def _rand(rng, shape, dt):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dt)


class _Once:
    """Complex sums that round the running value once per term.  Products are formed in
    a wider type and rounded where a fused multiply-add rounds."""

    def __init__(self, dt):
        self.S, self.W = (np.float32, np.float64) if dt == np.complex64 else (np.float64, np.longdouble)

    def r(self, v):
        return v.astype(self.S).astype(self.W)

    def parts(self, a):
        return a.real.astype(self.W), a.imag.astype(self.W)

    def mul(self, a, y):
        return self.r(a[0] * y[0] - self.r(a[1] * y[1])), self.r(a[0] * y[1] + self.r(a[1] * y[0]))

    def sub(self, x, p):
        return self.r(x[0] - p[0]), self.r(x[1] - p[1])


def _solve_once(Lw, B):
    """L^-1 B, unit lower; [matrix][row][column]."""
    o = _Once(B.dtype)
    l, x = o.parts(Lw), [v.copy() for v in o.parts(B)]
    for j in range(Lw.shape[-1] - 1):
        p = o.mul([c[:, j + 1:, j, None] for c in l], [c[:, j, None, :] for c in x])
        x[0][:, j + 1:], x[1][:, j + 1:] = o.sub([c[:, j + 1:] for c in x], p)
    return x[0] + 1j * x[1]


def _lu_once(A, ipiv):
    """The factors of A with the interchanges ipiv."""
    o = _Once(A.dtype)
    a = [v.copy() for v in o.parts(A)]
    b, n, _ = A.shape
    i = np.arange(b)
    for k in range(n):
        for c in a:
            c[i, k], c[i, ipiv[:, k]] = c[i, ipiv[:, k]].copy(), c[i, k].copy()
        re, im = a[0][:, k, k], a[1][:, k, k]
        den = o.r(re * re + o.r(im * im))
        inv = [o.r(re / den)[:, None], o.r(-im / den)[:, None]]
        a[0][:, k + 1:, k], a[1][:, k + 1:, k] = o.mul([c[:, k + 1:, k] for c in a], inv)
        p = o.mul([c[:, k + 1:, k, None] for c in a], [c[:, k, None, k + 1:] for c in a])
        t = o.sub([c[:, k + 1:, k + 1:] for c in a], p)
        a[0][:, k + 1:, k + 1:], a[1][:, k + 1:, k + 1:] = t
    return a[0] + 1j * a[1]


def _rms(r):
    return float(np.sqrt(np.mean(np.abs(r) ** 2)))


# Means over 64 matrices of 32 x 32 entries and more: their relative spread is below 1 %,
# and a second rounding per term adds 9 % and more.
@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_solve_rounds_once_per_term(probe, dt):
    L, ctx = probe
    rng = np.random.default_rng(32)
    b, n, nr = 64, 32, 64
    Lm = np.tril(_rand(rng, (b, n, n), dt) * dt(0.3), -1) + np.eye(n, dtype=dt)
    B = _rand(rng, (b, n, nr), dt)
    F = Lm.transpose(0, 2, 1).copy(order="C")  # U = I: the upper solve changes nothing
    X = B.transpose(0, 2, 1).copy(order="C")
    f = L.qbt_trsm_c64 if dt == np.complex64 else L.qbt_trsm_c128
    assert f(ctx, n, _p(F), _p(X), nr, b) == 0

    def err(x):
        return _rms(B.astype(np.clongdouble) - Lm.astype(np.clongdouble) @ x.astype(np.clongdouble))
    assert err(X.transpose(0, 2, 1)) <= 1.03 * err(_solve_once(Lm, B))


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
def test_factors_round_once_per_term(probe, dt):
    L, ctx = probe
    rng = np.random.default_rng(33)
    b, n = 64, 32
    A = _rand(rng, (b, n, n), dt)
    F, ipiv = A.transpose(0, 2, 1).copy(order="C"), np.zeros((b, n), np.int32)
    f = L.qbt_getrf_c64 if dt == np.complex64 else L.qbt_getrf_c128
    assert f(ctx, n, _p(F), _p(ipiv), b) == 0

    def err(lu):
        lu = lu.astype(np.clongdouble)
        r = np.tril(lu, -1) @ np.triu(lu) + np.triu(lu)
        return _rms(np.stack([A[i][_order(ipiv[i])] for i in range(b)]) - r)
    assert err(F.transpose(0, 2, 1)) <= 1.03 * err(_lu_once(A, ipiv))


def _order(ipiv):
    o = np.arange(len(ipiv))
    for s, q in enumerate(ipiv):
        o[s], o[q] = o[q], o[s]
    return o


@pytest.mark.parametrize("dt", [np.complex64, np.complex128])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (3, 63), (4, 64), (5, 65), (31, 64), (32, 1), (32, 65)])
def test_solves_at_their_edges(probe, dt, lower, n, nrhs):
    """Lower and upper solves one at a time against products in extended precision:
    |b - T x| <= 4 (n + 4) u |T||x| entry by entry (a term: four roundings of its parts
    and one of the sum; the reciprocal of a diagonal entry and its product: eight)."""
    L, ctx = probe
    u = np.finfo(dt).eps / 2
    rng = np.random.default_rng(n + nrhs)
    b = 5
    T = _rand(rng, (b, n, n), dt)
    T = np.tril(T, -1) + np.eye(n, dtype=dt) if lower else np.triu(T) + 4 * np.eye(n, dtype=dt)
    B = _rand(rng, (b, n, nrhs), dt)
    F, X = T.transpose(0, 2, 1).copy(order="C"), B.transpose(0, 2, 1).copy(order="C")
    f = L.qbt_trsm_c64 if dt == np.complex64 else L.qbt_trsm_c128
    assert f(ctx, n, _p(F), _p(X), nrhs, b) == 0
    x = X.transpose(0, 2, 1).astype(np.clongdouble)
    t = T.astype(np.clongdouble)
    assert np.all(np.abs(B - t @ x) <= 4 * (n + 4) * u * (np.abs(t) @ np.abs(x)))


# one row more than the leaf of four waves takes, the most of eight waves, one row more
@pytest.mark.parametrize("n", [4097, 8192, 8193])
def test_long_panel(probe, n):
    """A panel P^T L U with sparse dyadic factors, whose sums are exact and whose pivots
    are unique: both come back bit for bit."""
    L, ctx = probe
    rng = np.random.default_rng(n)
    w, unit = 512, np.array([1, -1, 1j, -1j])
    i, j = rng.integers(0, n, 6 * n), rng.integers(0, w, 6 * n)
    low, upp = i > j, (i < j) & (i < w)
    Lm = np.zeros((n, w), complex)
    Um = np.zeros((w, w), complex)
    Lm[i[low], j[low]] = rng.choice([0.5, 0.25], low.sum()) * rng.choice(unit, low.sum())
    Um[i[upp], j[upp]] = rng.choice([1.0, 2.0], upp.sum()) * rng.choice(unit, upp.sum())
    d = np.arange(w)
    Lm[d, d] = 1
    Um[d, d] = rng.choice([4.0, 8.0], w) * rng.choice(unit, w)
    perm = rng.permutation(n)
    A = np.empty((w, n), complex)  # [column][row]; row perm[i] is row i of L U
    A[:, perm] = (sp.csr_matrix(Lm) @ sp.csr_matrix(Um)).toarray().T
    ipiv = np.zeros(w, np.int32)
    assert L.qbt_first_panel_c128(ctx, n, w, _p(A), _p(ipiv)) == 0
    order = np.arange(n)
    for s, q in enumerate(ipiv):
        order[s], order[q] = order[q], order[s]
    assert np.array_equal(order[:w], perm[:w])
    inv = np.argsort(perm)
    ref = Lm[inv[order]]
    ref[:w] = np.tril(ref[:w], -1) + Um
    assert np.array_equal(A.T, ref)
