"""Each wavenumber of a call takes its own route (envelope tables where they stand in for
tables of the sizes given, else those): a matrix is the same bits whatever else is in the
list, and in whatever batches residuals are formed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
# tables that resolve H and J to 1e-12 at |k| = 14 and not at 700
CP = dict(n_panels_h=1500, M_h=9, n_panels_j=900, M_j=9)
FINE, COARSE = [14.0 + 0.2j, 13.7 - 0.4j, 14.1], [700.0 + 0.1j, 650.0, 700.3 - 0.2j]
LISTS = [[COARSE[0], FINE[0]], [FINE[0], COARSE[0], COARSE[1], FINE[1]], FINE[:2] + COARSE[:1] + FINE[2:]]


def _star(N=130, sym=None):
    import qbhip as q
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solver = q.CFIE_kress(10.0, b, symmetry=sym)
    return q, solver, q.evaluate_points(solver, b, 14.0, N=[N])


def test_the_list_has_both_routes(monkeypatch):
    q, solver, pts = _star()
    T = q.assemble(solver, pts, [FINE[0], COARSE[0]], **CP)
    monkeypatch.setenv("QB_ASM_TABLES", "1")
    t = q.assemble(solver, pts, [FINE[0], COARSE[0]], **CP)
    assert not np.array_equal(T[0], t[0]) and np.array_equal(T[1], t[1])


@pytest.mark.parametrize("z", LISTS)
def test_matrices(z):
    q, solver, pts = _star()
    T = q.assemble(solver, pts, z, **CP)
    for i, zi in enumerate(z):
        assert np.array_equal(T[i], q.assemble(solver, pts, [zi], **CP)[0])


@pytest.mark.parametrize("z", LISTS)
def test_derivatives(z):
    q, solver, pts = _star()
    T = q.assemble_with_derivatives(solver, pts, z, **CP)
    for i, zi in enumerate(z):
        for a, b in zip(T, q.assemble_with_derivatives(solver, pts, [zi], **CP)):
            assert np.array_equal(a[i], b[0])


@pytest.mark.parametrize("z", LISTS)
def test_residuals_in_any_batches(z):
    q, solver, pts = _star()
    rng = np.random.default_rng(1)
    phi = np.asfortranarray(rng.standard_normal((130, len(z))) + 1j * rng.standard_normal((130, len(z))))
    g = q.Geometry(pts, solver=solver)
    all_at_once = q.residual_norms(solver, pts, z, phi, geom=g, **CP)
    for batch in (1, 2):
        for a, b in zip(all_at_once, q.residual_norms(solver, pts, z, phi, geom=g, batch=batch, **CP)):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("z", LISTS)
def test_without_allocation(z):
    from test_zz_no_alloc import _hip, _noalloc
    q, solver, pts = _star()
    T, _ = _noalloc(q, solver, pts, z, CP, _hip())
    assert np.array_equal(T, q.assemble(solver, pts, z, **CP))


@pytest.mark.parametrize("centres", [[14.0, 700.0], [700.0, 14.0, 690.0]])
def test_windows_of_several_irreps(centres):
    """T of a mixed window stays as assembled; its matrices stand irrep by irrep."""
    import qbhip as q
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solvers = [q.CFIE_kress(10.0, b, symmetry=q.Rotation(5, m)) for m in range(3)]
    pts = q.evaluate_points(solvers[0], b, 14.0, N=[350])
    g = q.Geometry(pts, solver=solvers[0], irreps=solvers)
    nq = 4

    def matrices(k0):
        w = q.Window(solvers[0], pts, k0, 0.4, nq, precision="mixed", geom=g, **CP)
        T = np.array([w.matrix_cols(j, 0, 70) for j in range(nq * np.size(k0) * 3)])
        w.close()
        return T.reshape(3, np.size(k0), nq, 70, 70)
    T = matrices(np.array(centres))
    for i, k0 in enumerate(centres):
        assert np.array_equal(T[:, i], matrices(np.array([k0]))[:, 0])
