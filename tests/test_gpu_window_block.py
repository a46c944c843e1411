"""The block that a window's LU takes for its residues serves its moment solutions as
well: one allocation of several gigabytes per window fewer, given back with the window."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N, NQ = 4096, 4
CP = dict(n_panels_h=9000, M_h=9, n_panels_j=4000, M_j=9)


@pytest.fixture()
def disk():
    """A context that caches nothing, as the serving loop's."""
    import qbhip as q
    ctx = q.Context()
    ctx.set_cache_limit(0)
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solver = q.CFIE_kress(10.0, b)
    pts = q.evaluate_points(solver, b, 330.0, N=[N])
    geom = q.Geometry(pts, ctx, solver)

    made = []

    def window(k0=330.0):
        made.append(q.Window(solver, pts, k0, 0.4, NQ, geom=geom, **CP))
        return made[-1]
    yield q, ctx, window
    for w in made:  # before the context that they belong to
        w.close()
    geom.close()
    ctx.close()


def _probes(r, seed=3):
    rng = np.random.default_rng(seed)
    return np.asfortranarray(rng.standard_normal((N, r)) + 1j * rng.standard_normal((N, r)))


def test_one_block_for_residues_and_solutions(disk):
    q, ctx, window = disk
    free = ctx.device_bytes()
    ctx.set_residue_buffers(False)
    w = window()
    core = ctx.device_bytes() - free
    plain = w.moments(_probes(32))
    w.close()
    assert ctx.device_bytes() == free
    ctx.set_residue_buffers(True)
    w = window()
    block = ctx.device_bytes() - free - core
    assert block > 2 * 16 * NQ * N * 512  # the residues of 512 columns: 32 bytes an entry
    got = w.moments(_probes(32))
    assert ctx.device_bytes() == free + core + block
    w2 = window(331.0)  # the block is the context's: one for all its windows
    assert ctx.device_bytes() == free + 2 * core + block
    for a, b in zip(got, w.moments(_probes(32))):
        assert np.array_equal(a, b)
    # the two routes of the LU differ in rounding: backward errors of 1e-13 and less
    # against solutions that differ by the condition number times that
    for a, b in zip(got, plain):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    # solutions that do not fit take memory of their own, in the block's place
    r = block // (16 * NQ * N) + 1
    big = w.moments(_probes(r))
    assert ctx.device_bytes() == free + 2 * core
    small = w.moments(_probes(r)[:, :32])
    for a, b, c in zip(small, w.moments(_probes(r)[:, :32]), big):
        assert np.array_equal(a, b) and np.linalg.norm(a - c[:, :32]) <= 1e-11 * np.linalg.norm(a)
    w.close()
    w2.close()
    assert ctx.device_bytes() == free


def test_within_the_footprint(disk):
    """What a window holds while its moments are solved is what admission counted."""
    from qbhip.beyn import footprint
    q, ctx, window = disk
    free = ctx.device_bytes()
    for r in (8, 64, 256):
        w = window()
        # V, two moments and the QR block of 2 r columns stand beside the block
        held = ctx.device_bytes() - free + 5 * 16 * N * r
        w.moments_qr(_probes(r))
        w.close()
        assert held <= footprint(N, NQ, "fp64", r)
