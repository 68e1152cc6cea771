"""Pairs close to the surfaces (closed forms) and away, against the oracle: calls so small that one kernel takes all
pairs, up to 1e7 in FP64 and 2e6 in mixed precision, over triangles, planar elements with wires, and a mesh smaller than a
cluster; and the culled near pass of larger calls at the sizes where it changes the number of wavefronts that share
a group of 64 points (16 up to 512 groups, 4 up to 4,096, 1 above), over triangles, planar elements with wires, and
axisymmetric ones with both."""
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


def meshes(name):
    if name == "triangles":
        return G.cube_mesh(2)
    if name == "one":
        return G.cube_mesh(1).subset([0])
    wire = G.line_records([[-0.2, -0.2, 0.7]], [[0.3, 0.2, 0.8]], 2e-3)
    line = G.Mesh(np.full(1, G.LINESEGMENT, np.int32), wire, np.zeros(1, np.int32), np.zeros(1), np.zeros(1),
                  np.zeros(1, np.int32))
    return G.concat(G.cube_rect_mesh(2), G.cube_mesh(1, edge=0.5), line)


@pytest.mark.parametrize("name,npts", [("one", 1), ("one", 65), ("triangles", 64), ("triangles", 32768),
                                       ("triangles", 32769), ("triangles", 262145), ("mixed", 63),
                                       ("mixed", 32769)])
def test_near_pass_wavefronts(ctx, oracle, name, npts):
    """Small calls but for 48 triangles at 262,145 points, where the near pass has one wavefront per group."""
    from kassiopeia_amd import kemfield as K

    m = meshes(name)
    cont = K.KSurfaceContainer(ctx, m)
    sigma = np.random.default_rng(npts).normal(size=m.n) * 1e-9
    pts = G.points_shell(npts, 0.87, 1.6, npts)
    pts[0] = [0.5, 0.13, 0.07]  # in the plane of a face
    E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma).ElectricFieldAndPotential(pts)
    phr, Er = oracle.field(m.shapes, m.recs, sigma, pts)
    # FP64 sums of a few hundred terms in another order: far inside the 1e-12 that the field tests hold
    assert np.abs(phi - phr).max() <= 1e-12 * np.abs(phr).max()
    assert np.linalg.norm(E - Er, axis=1).max() <= 1e-12 * np.linalg.norm(Er, axis=1).max()
    cont.close()


@pytest.mark.parametrize("precision,n,npts", [("fp64", 1, 1), ("fp64", 5, 63), ("fp64", 47, 65), ("fp64", 48, 4097),
                                              ("mixed", 48, 130), ("mixed", 48, 41666), ("mixed", 48, 41667),
                                              ("fp64", 48, 208333), ("fp64", 48, 208334)])
def test_small_calls(ctx, oracle, precision, n, npts):
    """Both sides of the sizes up to which one kernel takes all pairs (1e7 pairs FP64, 2e6 mixed), ragged ranges and
    groups, a single element and point."""
    from kassiopeia_amd import kemfield as K

    m = meshes("triangles").subset(np.arange(n))
    cont = K.KSurfaceContainer(ctx, m)
    sigma = 1e-9 * np.random.default_rng(n).uniform(0.5, 1.5, size=m.n)
    pts = G.points_shell(npts, 0.87, 1.6, npts)
    E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma, precision).ElectricFieldAndPotential(pts)
    phr, Er = oracle.field(m.shapes, m.recs, sigma, pts)
    tol = 1e-12 if precision == "fp64" or n * npts <= 2e6 else 1e-6  # the mixed bar where FP32 pairs are taken
    assert np.abs(phi - phr).max() <= tol * np.abs(phr).max()
    assert np.linalg.norm(E - Er, axis=1).max() <= tol * np.linalg.norm(Er, axis=1).max()
    cont.close()


def larger_mesh(name):
    """320 to 1,535 elements: more pairs than a small call from 32,768 points on, fewer elements than the hierarchical pass."""
    if name == "triangles":
        return G.cube_mesh(6)
    parts = [G.cube_rect_mesh(7), G.cube_mesh(2, edge=0.5)]
    wires = G.line_records([[-0.2, -0.2, 0.7], [0.8, -0.4, 0.1]], [[0.3, 0.2, 0.8], [0.8, 0.4, 0.2]], 2e-3)
    kinds = [(G.LINESEGMENT, wires)]
    if name == "axisymmetric":
        kinds += [(G.CONICSECTION, G.conic_records([2.0, 2.5], [-1.0, 1.0], [2.5, 2.0], [1.0, 1.5])),
                  (G.RING, G.ring_records([2.2], [-1.5]))]
    for shape, recs in kinds:
        k = len(recs)
        parts.append(G.Mesh(np.full(k, shape, np.int32), recs, np.zeros(k, np.int32), np.zeros(k), np.zeros(k),
                            np.zeros(k, np.int32)))
    return G.concat(*parts)


@pytest.mark.parametrize("name", ["triangles", "planar", "axisymmetric"])
@pytest.mark.parametrize("npts", [32768, 32769, 262145])
def test_near_pass_past_small_calls(ctx, oracle, name, npts):
    from kassiopeia_amd import kemfield as K

    m = larger_mesh(name)
    assert m.n * npts > 1e7 and m.n < 1536
    cont = K.KSurfaceContainer(ctx, m)
    sigma = np.random.default_rng(npts).normal(size=m.n) * 1e-9
    pts = G.points_shell(npts, 0.87, 1.6, npts)
    pts[0] = [0.5, 0.13, 0.07]  # in the plane of a face
    E, phi = K.KIntegratingElectrostaticFieldSolver(cont, sigma).ElectricFieldAndPotential(pts)
    some = np.unique(np.concatenate([[0, npts - 1], np.random.default_rng(1).integers(0, npts, 1500)]))
    phr, Er = oracle.field(m.shapes, m.recs, sigma, pts[some], threads=8)
    # FP64 sums of a few hundred terms in another order: far inside the 1e-12 that the field tests hold
    assert np.abs(phi[some] - phr).max() <= 1e-12 * np.abs(phr).max()
    assert np.linalg.norm(E[some] - Er, axis=1).max() <= 1e-12 * np.linalg.norm(Er, axis=1).max()
    cont.close()
