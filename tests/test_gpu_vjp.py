"""The field term of the adjoint at the sizes where its kernel changes: points and elements around a wavefront, a round
of 256 points and several splits, points that mix the three rules and near pairs within one wavefront, against the
same derivative point by point (one call per point, summed on the host)."""
import numpy as np
import pytest

from kassiopeia_amd import geometry as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from kassiopeia_amd import kemfield as K

    c = K.Context(0)
    c.set_integrator("numeric")
    yield c
    c.close()


def vjp(ctx, cont, sigma, pts, g):
    n = sigma.size
    ds, dv = np.zeros(n), np.zeros((n, 9))
    p = lambda a: a.ctypes.data  # noqa: E731
    pts, g = np.ascontiguousarray(pts), np.ascontiguousarray(g)
    ctx.check(ctx.lib.kem_field_vjp(ctx.h, cont.h, p(sigma), len(pts), p(pts), p(g), p(ds), p(dv)))
    return ds, dv


@pytest.mark.parametrize("n,npts", [(1, 1), (63, 64), (64, 65), (65, 255), (192, 257), (300, 300)])
def test_field_vjp_splits(ctx, n, npts):
    from kassiopeia_amd import kemfield as K

    m = G.cube_mesh(5).subset(np.arange(n))  # 300 triangles of 0.2: sizes about 0.23
    cont = K.KSurfaceContainer(ctx, m)
    rng = np.random.default_rng(n + npts)
    sigma = rng.normal(size=n) * 1e-9
    # shells from the closed forms (0.8 m) past the 7-point rule (131 sizes, 30 m)
    pts = np.concatenate([G.points_shell(npts, a, b, npts) for a, b in
                          ((0.6, 0.9), (1.0, 5.0), (5.0, 25.0), (25.0, 60.0))])[rng.permutation(4 * npts)[:npts]]
    g = rng.normal(size=npts)
    ds, dv = vjp(ctx, cont, sigma, pts, g)
    one = [vjp(ctx, cont, sigma, pts[k:k + 1], g[k:k + 1]) for k in range(npts)]
    rs, rv = sum(o[0] for o in one), sum(o[1] for o in one)
    # the same rules to their 1e-15 truncation, sums of up to 300 terms in another order
    assert np.abs(ds - rs).max() <= 1e-13 * np.abs(rs).max()
    assert np.abs(dv - rv).max() <= 1e-12 * np.abs(rv).max()
    cont.close()


def test_field_vjp_chunks(ctx):
    """Enough pairs for chunks of 64 points, and a ragged last one, against batches of 125 points (chunks of a few)."""
    from kassiopeia_amd import kemfield as K

    m = G.cube_mesh(21)  # 5,292 triangles of 0.05: sizes about 0.06
    cont = K.KSurfaceContainer(ctx, m)
    rng = np.random.default_rng(11)
    npts = 7013
    sigma = rng.uniform(0.5, 1.0, size=m.n) * 1e-9
    pts = np.concatenate([G.points_shell(npts, a, b, npts) for a, b in ((0.45, 0.9), (0.9, 3.0), (3.0, 20.0))])
    pts = pts[rng.permutation(len(pts))[:npts]]
    g = rng.uniform(0.5, 1.0, size=npts)
    ds, dv = vjp(ctx, cont, sigma, pts, g)
    parts = [vjp(ctx, cont, sigma, pts[k:k + 125], g[k:k + 125]) for k in range(0, npts, 125)]
    rs, rv = sum(o[0] for o in parts), sum(o[1] for o in parts)
    # sums of 7,013 terms in another order: 7,013 x 2^-53 = 8e-13 of the sum of magnitudes, which for the densities'
    # positive terms is the sum, and for the vertices' at most ten times the largest
    assert np.abs(ds - rs).max() <= 1e-12 * np.abs(rs).max()
    assert np.abs(dv - rv).max() <= 1e-11 * np.abs(rv).max()
    cont.close()
