"""The hierarchical far field against the flat passes: fields at many points (hierarchical) and at batches of fewer than 4,096 of
the same points (always flat), over meshes of triangles, of rectangles with wires and of symmetry groups, element counts
that leave the last run partial, point counts around one and two points per lane and with ragged last groups, smooth
densities and densities of random sign, and point sets that are hard to group: scattered clumps, one point many times,
points far away, points that are not finite."""
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


def mesh_of(kind, n):
    if kind == "triangles":
        m = G.coax_mesh(nphi_in=24, nphi_out=48, nz=31, ncap_r=4, ncap_phi=33)
        return m.subset(np.arange(min(n, m.n)))
    if kind == "frame":
        k = ((n - 40) / 6) ** 0.5
        rect = G.cube_rect_mesh(int(k))
        w = n - rect.n
        x = np.linspace(-0.5, 0.5, w)
        p0 = np.stack([x, np.full(w, -0.5), np.full(w, 0.8)], 1)
        wires = G.line_records(p0, p0 + np.array([0.0, 1.0, 0.1]), 1e-4)
        return G.concat(rect, G.Mesh(np.full(w, G.LINESEGMENT, np.int32), wires, np.zeros(w, np.int32), np.zeros(w),
                                     np.zeros(w), np.zeros(w, np.int32)))
    return G.mirror_groups(G.cube_mesh(round((n / 24) ** 0.5)), [0.0, 0.0, 1.5], [0.0, 0.0, 1.0])


def points_of(kind, npts, seed):
    if kind == "triangles":
        return G.points_annulus(npts, 0.51, 0.99, 1.95, seed)
    return G.points_shell(npts, 0.9, 2.5, seed)


def flat(cont, sigma, pts, precision):
    from kassiopeia_amd import kemfield as K

    s = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision)
    E, phi = zip(*[s.ElectricFieldAndPotential(pts[i:i + 4000]) for i in range(0, len(pts), 4000)])
    return np.concatenate(E), np.concatenate(phi)


@pytest.mark.parametrize("kind,n,npts,rough", [
    ("triangles", 4007, 16001, False), ("triangles", 4007, 65536, True), ("triangles", 4007, 65537, True),
    ("triangles", 3001, 65601, False), ("frame", 3219, 40001, True), ("frame", 3219, 131077, False),
    ("groups", 4800, 33000, True)])
def test_tree_against_flat(ctx, kind, n, npts, rough):
    from kassiopeia_amd import kemfield as K

    m = mesh_of(kind, n)
    cont = K.KSurfaceContainer(ctx, m)
    rng = np.random.default_rng(n + npts)
    c = m.centroids()
    sigma = 1e-9 * (rng.normal(size=m.n) if rough else 1.0 + 0.5 * np.sin(3.0 * c[:, 2] + c[:, 0]))
    pts = points_of(kind, npts, npts)
    some = np.unique(np.concatenate([[0, npts - 1], rng.integers(0, npts, 6000)]))
    E0, p0 = flat(cont, sigma, pts[some], "fp64")
    for precision, tol in (("fp64", 1e-13), ("mixed", 1e-6)):
        E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision).ElectricFieldAndPotential(pts)
        # FP64: expansions to 6e-15 of each run's field and the pairs' own rules to 3e-14; mixed: its bar
        assert np.linalg.norm(E[some] - E0) <= tol * np.linalg.norm(E0), precision
        assert np.linalg.norm(phi[some] - p0) <= tol * np.linalg.norm(p0), precision
        assert np.abs(phi[some] - p0).max() <= 10 * tol * np.abs(p0).max(), precision
    cont.close()


def test_tree_hard_points(ctx):
    from kassiopeia_amd import kemfield as K

    m = mesh_of("triangles", 4007)
    cont = K.KSurfaceContainer(ctx, m)
    sigma = 1e-9 * np.random.default_rng(3).normal(size=m.n)
    rng = np.random.default_rng(4)
    clumps = rng.uniform(-2.0, 2.0, (40, 3))[rng.integers(0, 40, 30000)] + 1e-3 * rng.normal(size=(30000, 3))
    sets = {"clumps": clumps, "one": np.tile([[0.7, 0.1, 0.2]], (20000, 1)),
            "far": np.concatenate([clumps, 1e5 * rng.normal(size=(50, 3)), m.centroids()[:500]])}
    for name, pts in sets.items():
        E0, p0 = flat(cont, sigma, pts[::7], "fp64")
        E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, "fp64").ElectricFieldAndPotential(pts)
        assert np.linalg.norm(E[::7] - E0) <= 1e-13 * np.linalg.norm(E0), name
        assert np.linalg.norm(phi[::7] - p0) <= 1e-13 * np.linalg.norm(p0), name
    # points that are not finite give values that are not, and leave the others alone
    pts = clumps.copy()
    pts[[5, 77]] = np.nan
    pts[[123, 20000], 1] = np.inf
    bad = ~np.isfinite(pts).all(1)
    E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, "fp64").ElectricFieldAndPotential(pts)
    E0, p0 = flat(cont, sigma, clumps[::7], "fp64")
    ok = ~bad[::7]
    assert not np.isfinite(phi[np.isnan(pts).any(1)]).any()
    assert np.linalg.norm(E[::7][ok] - E0[ok]) <= 1e-13 * np.linalg.norm(E0[ok])
    assert np.linalg.norm(phi[::7][ok] - p0[ok]) <= 1e-13 * np.linalg.norm(p0[ok])
    cont.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("npts", [16384, 70000])
@pytest.mark.parametrize("lane", [5, 31, 32, 60, 62, 63])
def test_tree_points_that_are_not_finite(ctx, lane, npts, precision):
    """One coordinate of one point in each second group not a number, in lanes of both halves of a wavefront, with one and two
    points per lane: alone, so that the others stay in curve order, and beside an infinite coordinate, which leaves all
    points in the caller's order, where every second one lies far from its neighbours."""
    from kassiopeia_amd import kemfield as K

    m = mesh_of("triangles", 4007)
    cont = K.KSurfaceContainer(ctx, m)
    sigma = 1e-9 * np.random.default_rng(5).normal(size=m.n)
    tol = 1e-13 if precision == "fp64" else 1e-6  # as for finite points
    for infinite in (False, True):
        pts = points_of("triangles", npts, 6)
        pts[lane::128, 0] = np.nan
        if infinite:
            pts[1::2] = 0.0
            pts[lane::128, 0] = np.nan
            pts[npts // 2, 1] = np.inf
        some = np.unique(np.concatenate([np.arange(npts // 2 - 64, npts // 2 + 64), np.arange(0, npts, 5)]))
        E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision).ElectricFieldAndPotential(pts)
        E0, p0 = flat(cont, sigma, pts[some], "fp64")
        ok = np.isfinite(pts[some]).all(1)
        E, phi = E[some], phi[some]
        assert not np.isfinite(E[np.isnan(pts[some]).any(1)]).any()
        assert np.linalg.norm(E[ok] - E0[ok]) <= tol * np.linalg.norm(E0[ok]), infinite
        assert np.linalg.norm(phi[ok] - p0[ok]) <= tol * np.linalg.norm(p0[ok]), infinite
    cont.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,n", [("triangles", 4992), ("frame", 3219), ("cube", 3072)])
def test_tree_one_charged_element(ctx, kind, n, precision):
    """One charged element at a time, where the coefficients of the expansions of a run that has it at its rim do not decay:
    clumps of points all around it, where runs are taken near and far, point by point."""
    from kassiopeia_amd import kemfield as K

    m = G.cube_mesh(16) if kind == "cube" else mesh_of(kind, n)
    cont = K.KSurfaceContainer(ctx, m)
    c = m.centroids()
    size = np.ptp(c, axis=0).max()
    # each run's terms are omitted below 6e-15 (FP64) and 3e-7 (mixed) of the element's field at the point, and the rules of
    # the pairs err by up to 3e-14 (FP64, in either evaluation) and 4e-7 (mixed)
    tol = 6e-14 if precision == "fp64" else 6e-7
    for j in np.random.default_rng(n).integers(0, m.n, 24):
        rng = np.random.default_rng(j)
        sigma = np.zeros(m.n)
        sigma[j] = 1e-9
        out = rng.normal(size=(1100, 3))
        out *= (size * np.exp(rng.uniform(np.log(0.03), np.log(3.0), 1100)) / np.linalg.norm(out, axis=1))[:, None]
        pts = np.repeat(c[j] + out, 32, 0) + 1e-7 * rng.normal(size=(1100 * 32, 3))
        E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision).ElectricFieldAndPotential(pts)
        E0, p0 = flat(cont, sigma, pts, "fp64")
        assert (np.linalg.norm(E - E0, axis=1) / np.linalg.norm(E0, axis=1)).max() <= tol, j
        assert (np.abs(phi - p0) / np.abs(p0)).max() <= tol, j
    cont.close()


@pytest.mark.parametrize("n,npts,precision", [(36000, 20001, "fp64"), (64000, 20001, "mixed"), (140000, 8193, "fp64"),
                                              (240000, 8193, "mixed")])
def test_tree_coarser_lowest_runs(ctx, n, npts, precision):
    """Up to 65,536 points the lowest runs expanded hold 64 elements from about 33,000 (FP64) or 58,000 (mixed) on, and
    256 from four times as many: several rounds of 16 elements in each expansion, levels from the second or third on."""
    from kassiopeia_amd import kemfield as K

    m = G.ring_bore_mesh(n_target=n, volts=np.zeros(32))
    cont = K.KSurfaceContainer(ctx, m)
    rng = np.random.default_rng(n)
    pts = G.points_annulus(npts, 0.0, 1.88, 4.0, 7)
    some = np.unique(np.concatenate([[0, npts - 1], rng.integers(0, npts, 3000)]))
    tol = 1e-13 if precision == "fp64" else 1e-6  # as for runs of 16
    c = m.centroids()
    for sigma in (1e-9 * rng.normal(size=m.n), 1e-9 * (1.0 + 0.5 * np.sin(3.0 * c[:, 2] + c[:, 0]))):
        E0, p0 = flat(cont, sigma, pts[some], "fp64")
        E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision).ElectricFieldAndPotential(pts)
        assert np.linalg.norm(E[some] - E0) <= tol * np.linalg.norm(E0)
        assert np.linalg.norm(phi[some] - p0) <= tol * np.linalg.norm(p0)
    cont.close()


@pytest.mark.parametrize("kind,n,npts,sets,precision", [
    ("triangles", 4007, 40001, 4, "fp64"), ("frame", 3219, 262147, 24, "fp64"), ("groups", 4800, 33000, 3, "fp64"),
    ("triangles", 4007, 150001, 3, "mixed"), ("triangles", 4992, 262149, 6, "mixed"),
    ("frame", 3219, 300000, 5, "mixed")])
def test_tree_sets(ctx, kind, n, npts, sets, precision):
    """Points of several sets in one call, which the pass visits set by set: a set without points, one with a single
    point, runs of one set and alternating ones, groups of 64 points that hold the ends of several."""
    from kassiopeia_amd import kemfield as K

    m = mesh_of(kind, n)
    cont = K.KSurfaceContainer(ctx, m)
    rng = np.random.default_rng(n + npts)
    S = 1e-9 * rng.normal(size=(m.n, sets))
    pts = points_of(kind, npts, npts)
    which = np.repeat(rng.integers(2, sets, npts // 37 + 1), 37)[:npts]
    which[: npts // 5] = rng.integers(2, sets, npts // 5)
    which[npts // 2] = 1  # and none of set 0
    E, phi = K.field_sets(cont, S, which.astype(np.int32), pts, precision)
    tol = 1e-13 if precision == "fp64" else 1e-6  # as for one set
    for k in range(1, sets):
        some = np.flatnonzero(which == k)
        some = some[np.unique(np.concatenate([[0, len(some) - 1], rng.integers(0, len(some), 800)]))]
        E0, p0 = flat(cont, np.ascontiguousarray(S[:, k]), pts[some], "fp64")
        assert np.linalg.norm(E[some] - E0) <= tol * np.linalg.norm(E0), k
        assert np.linalg.norm(phi[some] - p0) <= tol * np.linalg.norm(p0), k
    cont.close()
