"""Matrices from the envelope tables that stand in for fine uniform tables, against
the same calls with the uniform tables (QB_ASM_TABLES=1), the general route."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CP = dict(n_panels_h=9000, M_h=9, n_panels_j=4000, M_j=9)  # errors of 1e-14: both routes resolve H and J
# Envelope and table values each lie within 1.5e-14 of |H| <= 5 (|k r| >= 0.2); the
# weights of an entry are at most 2 (k s w is 0.6 at ten nodes per wavelength, R_ij log
# terms double it): 2 * 2 * 5 * 1.5e-14 = 3e-13.  DLP values below |k r| = 0.2 come with
# H_1's size, 1 / (k r), which the test's shapes keep above 0.2.
TOL = 3e-13


def _solver(op, kind, Ns, k0):
    import qbhip as q
    b = {"star": lambda: q.make_star_polar_boundary(1.0, 0.2, 5), "ellipse": lambda: q.make_full_ellipse(1.0, 0.6),
         "circle_hole": lambda: q.CircularHoleBilliard(1.0, holes=[(0.3, 0.35, 0.0)])}[kind]()
    solver = (q.DLP_kress if op == "dlp" else q.CFIE_kress)(10.0, b)
    return q, solver, q.evaluate_points(solver, b, k0, N=Ns)


def _both(monkeypatch, f):
    got = f()
    monkeypatch.setenv("QB_ASM_TABLES", "1")
    ref = f()
    monkeypatch.delenv("QB_ASM_TABLES")
    return got, ref


# conjugate pairs in any order, real nodes, nodes without a partner, a near-real one,
# two nodes with one conjugate, and one wavenumber alone
LISTS = [[0.4 + 0.3j, -0.2 + 0.0j, 0.4 - 0.3j], [0.1 + 0.2j, 0.3 - 0.1j, -0.5 + 1e-12j, 0.2],
         [0.25 + 0.5j, 0.25 - 0.5j, 0.25 - 0.5j, 0.1j], [-0.3 - 0.4j], [0.0]]
GEOMS = [("cfie", "star", [130], 14.0), ("cfie", "circle_hole", [98, 45], 11.0), ("cfie", "star", [64], 7.0),
         ("dlp", "ellipse", [197], 21.0), ("dlp", "star", [63], 7.0)]


@pytest.mark.parametrize("dz", LISTS)
@pytest.mark.parametrize("op,kind,Ns,k0", GEOMS)
def test_matrices(monkeypatch, op, kind, Ns, k0, dz):
    q, solver, pts = _solver(op, kind, Ns, k0)
    z = k0 + np.array(dz)
    got, ref = _both(monkeypatch, lambda: q.assemble(solver, pts, z, **CP))
    assert not np.array_equal(got, ref)  # two routes
    assert np.max(np.abs(got - ref)) <= TOL


@pytest.mark.parametrize("dz", LISTS[:2])
@pytest.mark.parametrize("op,kind,Ns,k0", GEOMS)
def test_derivatives(monkeypatch, op, kind, Ns, k0, dz):
    """The derivatives carry the distance (at most 2.5) once and twice."""
    q, solver, pts = _solver(op, kind, Ns, k0)
    z = k0 + np.array(dz)
    got, ref = _both(monkeypatch, lambda: q.assemble_with_derivatives(solver, pts, z, **CP))
    for n, (a, b) in enumerate(zip(got, ref)):
        assert not np.array_equal(a, b)
        assert np.max(np.abs(a - b)) <= TOL * 2.5 ** n


def test_residuals(monkeypatch):
    q, solver, pts = _solver("cfie", "star", [150], 15.0)
    rng = np.random.default_rng(3)
    phi = rng.standard_normal((150, 5)) + 1j * rng.standard_normal((150, 5))
    phi = np.asfortranarray(phi / np.linalg.norm(phi, axis=0))
    z = 15.0 + np.array([0.3, -0.2 + 1e-12j, 0.1 - 1e-12j, 0.4j, 0.25])
    got, ref = _both(monkeypatch, lambda: q.residual_norms(solver, pts, z, phi, **CP))
    for a, b in zip(got, ref):
        # sums of up to 150 entries, each to TOL
        assert np.max(np.abs(np.asarray(a) - np.asarray(b))) <= 150 * TOL


@pytest.mark.parametrize("n_irr", [2, 3, 5])
def test_reduced_window(monkeypatch, n_irr):
    """T of a mixed window stays as assembled; entries are sums of five images."""
    import qbhip as q
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solvers = [q.CFIE_kress(10.0, b, symmetry=q.Rotation(5, m)) for m in range(n_irr)]
    pts = q.evaluate_points(solvers[0], b, 30.0, N=[350])
    g = q.Geometry(pts, solver=solvers[0], irreps=solvers)

    def cols():
        w = q.Window(solvers[0], pts, 30.0, 0.4, 6, precision="mixed", geom=g, **CP)
        T = [w.matrix_cols(j, 0, 70) for j in range(6 * n_irr)]
        w.close()
        return np.array(T)
    got, ref = _both(monkeypatch, cols)
    assert not np.array_equal(got, ref)
    assert np.max(np.abs(got - ref)) <= 5 * TOL


def test_coarse_tables_are_interpolated(monkeypatch):
    q, solver, pts = _solver("cfie", "star", [130], 14.0)
    cp = dict(n_panels_h=300, M_h=5, n_panels_j=100, M_j=5)
    got, ref = _both(monkeypatch, lambda: q.assemble(solver, pts, [14.0 + 0.2j], **cp))
    assert np.array_equal(got, ref)
