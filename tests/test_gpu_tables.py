"""Chebyshev tables of every degree and of panel counts around the number that a wave
builds at once, seen through the matrices assembled from them: the oracle builds the
same tables (coarse ones too: both interpolate, neither needs to be accurate)."""
import numpy as np
import pytest
import scipy.special as sp

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(op, kind, Ns, k0):
    import qbhip as q
    b = {"star": lambda: q.make_star_polar_boundary(1.0, 0.2, 5), "ellipse": lambda: q.make_full_ellipse(1.0, 0.6),
         "circle_hole": lambda: q.CircularHoleBilliard(1.0, holes=[(0.3, 0.35, 0.0)])}[kind]()
    solver = (q.DLP_kress if op == "dlp" else q.CFIE_kress)(10.0, b)
    return q, solver, q.evaluate_points(solver, b, k0, N=Ns)


# np_h, M_h, np_j, M_j: 64 / (M + 1) panels per wave, one more and one fewer, one
# panel in all, both kinds of one degree and of different ones
@pytest.mark.parametrize("cp", [(1, 2, 1, 16), (21, 2, 22, 3), (9, 6, 10, 5), (33, 5, 1, 7),
                                (7, 7, 8, 7), (3, 15, 5, 16), (401, 4, 150, 5), (64, 8, 63, 9)])
@pytest.mark.parametrize("op,kind,Ns,k0", [("cfie", "star", [130], 12.0),
                                           ("cfie", "circle_hole", [98, 46], 9.0),
                                           ("dlp", "ellipse", [194], 15.0)])
def test_matrices_from_tables(op, kind, Ns, k0, cp):
    """Every entry to 1e-12 of the largest table sample times its own weights:
    17 coefficients of 17 samples each and a Clenshaw sum round to below
    17 * 17 * 4 u = 1.3e-13 of max |H_1(z rmin)|; weights and k r are at most 1 and
    k0 times rmax = 3 in the entries."""
    q, solver, pts = _case(op, kind, Ns, k0)
    z = np.array([k0 + 0.4j, k0 - 0.3j, k0])
    T = q.assemble(solver, pts, z, n_panels_h=cp[0], M_h=cp[1], n_panels_j=cp[2], M_j=cp[3])
    comps = O.make_geometry(kind, Ns)
    ocp = O.ChebParams(*cp)
    ref = O.dlp_assemble(comps[0], z, ocp) if op == "dlp" else O.cfie_assemble(comps, z, ocp)
    x, y = (np.concatenate([getattr(c, f) for c in comps]) for f in "xy")
    r = np.hypot(x[:, None] - x, y[:, None] - y)
    rmin = np.min(r[r > 0])
    tol = 1e-12 * max(1.0, np.max(np.abs(sp.hankel1(1, z * rmin))))
    assert np.max(np.abs(T - ref)) <= tol
