"""Norms formed on the device, at row and column counts around the groups of 4, 16, 64
and 256 that the kernels take."""
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
