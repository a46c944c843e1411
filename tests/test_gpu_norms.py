"""Norms formed on the device, at row and column counts around the groups of 4, 16, 64
and 256 that the kernels take."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nl,batch", [(20, 1, 0), (63, 3, 2), (64, 2, 0), (65, 5, 3), (255, 2, 0), (257, 3, 2), (514, 2, 1)])
def test_residual_norms(N, nl, batch):
    """Against numpy's norms of the same matrices: sums of N terms round to below N u."""
    import qbhip as q
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solver = q.CFIE_kress(10.0, b)
    k0 = N / 12.0
    pts = q.evaluate_points(solver, b, k0, N=[N])
    rng = np.random.default_rng(N)
    z = k0 + rng.uniform(-0.3, 0.3, nl) + 0.05j * rng.standard_normal(nl)
    phi = np.asfortranarray(rng.standard_normal((N, nl)) + 1j * rng.standard_normal((N, nl)))
    cp = dict(n_panels_h=5000, M_h=7, n_panels_j=2000, M_j=7)
    got = q.residual_norms(solver, pts, z, phi, batch=batch, **cp)
    T = q.assemble(solver, pts, z, **cp)
    for i in range(nl):
        y, a = T[i] @ phi[:, i], np.abs(T[i])
        ref = [np.linalg.norm(y), np.abs(y).sum(), np.abs(y).max(), a.sum(0).max(), a.sum(1).max()]
        # a component of y rounds to below N u times the row sum of |T| |phi|
        tol = 4 * N * 1.2e-16 * (a @ np.abs(phi[:, i])).sum()
        for c in range(5):
            assert abs(got[c][i] - ref[c]) <= (tol if c < 3 else 4 * N * 1.2e-16 * ref[c])


@pytest.mark.parametrize("n,nb", [(1, 1), (3, 2), (4, 1), (15, 2), (17, 3), (63, 1), (65, 2), (130, 2), (300, 3)])
def test_matrix_norms(n, nb):
    import qbhip as q
    L = C.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libqbt_linalg.so"))
    rng = np.random.default_rng(n)
    A = rng.standard_normal((nb, n, n)) + 1j * rng.standard_normal((nb, n, n))
    rows, mx = np.zeros(nb), np.zeros(nb)
    assert L.qbt_node_norms(C.c_void_p(q.default_context().ptr.value), n, nb, C.c_void_p(A.ctypes.data),
                            C.c_void_p(rows.ctypes.data), C.c_void_p(mx.ctypes.data)) == 0
    # A[b] holds the matrix column by column
    assert np.allclose(rows, np.abs(A).sum(1).max(1), rtol=n * 2.3e-16, atol=0)
    assert np.allclose(mx, np.abs(A).max((1, 2)), rtol=2.3e-16, atol=0)
