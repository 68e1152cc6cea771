"""Matrix storage handed back to the context on kem_matrix_destroy and reused by the next
assembly of the same size: a matrix assembled into reused storage equals, bit for bit, the same
matrix assembled into fresh storage on another context (every entry rewritten, nothing of the
previous matrix left), in FP64, FP32 and BF16, with a matrix of another size in between.  Host-array
field calls: what they allocate beyond a few MiB goes back when they return."""
import ctypes

import numpy as np
import pytest

from kassiopeia_amd import geometry as G

pytestmark = pytest.mark.gpu


def _scaled(m, f):
    recs = m.recs.copy()
    recs[:, :2] *= f  # side lengths
    recs[:, 2:5] *= f  # first vertex
    return G.Mesh(m.shapes.copy(), recs, m.bc_type.copy(), m.bc_value.copy(), m.bc_flux.copy(), m.group.copy())


def test_matrix_storage_reuse():
    from kassiopeia_amd import kemfield as K

    m1 = G.cube_mesh(8)
    m2 = _scaled(m1, 1.5)
    mo = G.cube_mesh(6)  # another size
    ctx, fresh = K.Context(0), K.Context(0)
    try:
        X = np.random.default_rng(4).normal(size=(m1.n, 5))
        c1, c2, co = (K.KSurfaceContainer(ctx, m) for m in (m1, m2, mo))
        A1 = K.KBoundaryIntegralMatrix(c1, fp64=True, fp32=True, bf16=True)
        A1.to_numpy()
        A1.close()
        Ao = K.KBoundaryIntegralMatrix(co, fp64=True, fp32=True)
        A2 = K.KBoundaryIntegralMatrix(c2, fp64=True, fp32=True, bf16=True)  # the storage of A1
        Ao.close()
        f2 = K.KSurfaceContainer(fresh, m2)
        R2 = K.KBoundaryIntegralMatrix(f2, fp64=True, fp32=True, bf16=True)
        assert np.array_equal(A2.to_numpy(), R2.to_numpy())
        for prec in ("mixed", "bf16", "fp64"):
            assert np.array_equal(A2.MultiplyBatch(X, prec), R2.MultiplyBatch(X, prec)), prec
        A2.close()
        R2.close()
        for c in (c1, c2, co, f2):
            c.close()
    finally:
        ctx.close()
        fresh.close()


def _free_memory():
    """Bytes free on the device, from the runtime that the library is linked to."""
    from kassiopeia_amd import _lib

    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_host_field_calls_give_memory_back():
    from kassiopeia_amd import kemfield as K

    m = G.cube_mesh(4)
    ctx = K.Context(0)
    try:
        cont = K.KSurfaceContainer(ctx, m)
        solver = K.KIntegratingElectrostaticFieldSolver(cont, np.full(m.n, 1e-9))
        npts = 1_000_000  # 56 MB of points and results
        pts = G.points_shell(npts, 1.0, 2.0, 1)
        E, phi = solver.ElectricFieldAndPotential(pts)  # and the workspace of such calls, which stays
        few = solver.ElectricFieldAndPotential(pts[:1000])
        free = _free_memory()
        own = 8 * (m.n + 7 * npts)
        # the workspace through device arrays alone, on a context that never took host arrays
        other = K.Context(0)
        oc = K.KSurfaceContainer(other, m)
        S = K.DeviceArray(other, np.full(m.n, 1e-9))
        X = [K.DeviceArray(other, np.ascontiguousarray(pts[:, k])) for k in range(3)]
        O = [K.DeviceArray.empty(other, npts) for _ in range(4)]
        before = _free_memory()
        other.check(other.lib.kem_field_eval_device(other.h, oc.h, S.ptr, npts, X[0].ptr, X[1].ptr, X[2].ptr, 0,
                                                    O[0].ptr, O[1].ptr, O[2].ptr, O[3].ptr))
        other.sync()
        workspace = before - _free_memory()
        assert np.array_equal(np.stack([o.get() for o in O[1:]], 1), E) and np.array_equal(O[0].get(), phi)
        assert np.allclose(few[1], phi[:1000], rtol=1e-12)
        for a in X + O + [S]:
            a.close()
        oc.close()
        other.close()
        cont.close()
        ctx.close()
        ctx = None
        # what the host-array context still held: its workspace, and of the staging no more than 16 MiB (and as much slack
        # for the allocator's pages)
        held = _free_memory() - free
        assert held <= workspace + (32 << 20) < workspace + own
    finally:
        if ctx is not None:
            ctx.close()
