"""GMRES iterations at the sizes where their kernels change: rows per thread (1 below 32,768 rows, 2, 4 and 16 above,
doubling but for the last), a last chunk of one row, systems smaller than a chunk, more basis columns than a wavefront has
lanes, restarts; FP64 and FP32-matrix solves, and transposed ones, whose product is not left in parts, against a direct
solution."""
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


@pytest.mark.parametrize("n", [1, 2, 48, 255, 256, 257, 769])
def test_small_systems(ctx, n):
    from kassiopeia_amd import kemfield as K

    m = G.coax_mesh(nphi_in=8, nphi_out=12, nz=16, ncap_r=2, ncap_phi=18).subset(np.arange(n))
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont, fp64=True, fp32=True)
    b = np.random.default_rng(n).normal(size=n)
    ref = np.linalg.solve(A.to_numpy(), b)
    for precision, restart in (("fp64", 0), ("fp64", 37), ("mixed", 0)):
        x, st, rc = A.solve(b, tolerance=1e-11, restart=restart, precision=precision, max_iterations=4000)
        assert rc == 0 and st.true_residual <= 2e-11, (precision, restart)
        # a Krylov space has at most n dimensions; refinements and restarts each begin another
        assert st.iterations <= n or precision == "mixed" or restart
        if not restart:  # 1e-11 on the residual times the conditioning of these meshes (below 1e3)
            assert np.linalg.norm(x - ref) <= 1e-7 * np.linalg.norm(ref), precision
    A.close()
    cont.close()


@pytest.mark.parametrize("n", [1, 2, 255, 257, 769])
def test_transposed(ctx, n):
    import ctypes

    from kassiopeia_amd import _lib
    from kassiopeia_amd import kemfield as K

    m = G.coax_mesh(nphi_in=8, nphi_out=12, nz=16, ncap_r=2, ncap_phi=18).subset(np.arange(n))
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont, fp64=True, fp32=True)
    b = np.random.default_rng(n).normal(size=n)
    ref = np.linalg.solve(A.to_numpy().T, b)
    for precision, restart in ((_lib.KEM_FP64, 0), (_lib.KEM_FP64, 37), (_lib.KEM_MIXED, 0)):
        o, st, x = _lib.SolveOpts(), _lib.SolveStats(), np.zeros(n)
        ctx.lib.kem_solve_opts_default(ctypes.byref(o))
        o.method, o.precision, o.tolerance, o.restart, o.max_iterations = \
            _lib.KEM_SOLVER_GMRES, precision, 1e-11, restart, 4000
        rc = ctx.lib.kem_solve_transposed(A.h, ctypes.byref(o), K._ptr(b), K._ptr(x), ctypes.byref(st))
        assert rc == 0 and st.true_residual <= 2e-11, (precision, restart)
        assert np.linalg.norm(A.MultiplyTranspose(x) - b) <= 2e-11 * np.linalg.norm(b)
        if not restart:  # as for the solves of A
            assert np.linalg.norm(x - ref) <= 1e-7 * np.linalg.norm(ref), precision
    A.close()
    cont.close()


@pytest.mark.parametrize("n", [66000, 131100])
def test_rows_per_thread(n):
    """4 and 16 rows per thread (35 and 137 GB of FP64 matrix, given back with the context)."""
    from kassiopeia_amd import kemfield as K

    ctx = K.Context(0)
    ctx.set_integrator("numeric")
    m = G.ring_bore_mesh(n_target=n, volts=np.linspace(-1000.0, -10.0, 32))
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont)
    print(f"{n} unknowns assembled", flush=True)
    x, st, rc = A.solve(cont.rhs(), tolerance=1e-10)
    assert rc == 0 and st.true_residual <= 2e-10
    b = cont.rhs()
    assert np.linalg.norm(A.Multiply(x) - b) <= 2e-10 * np.linalg.norm(b)
    A.close()
    cont.close()
    ctx.close()


def test_many_rows(ctx):
    """33,000 unknowns: two rows per thread (8.7 GB of FP64 matrix)."""
    from kassiopeia_amd import kemfield as K

    m = G.ring_bore_mesh(n_target=33000, volts=np.linspace(-1000.0, -10.0, 32))
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont)
    x, st, rc = A.solve(cont.rhs(), tolerance=1e-10)
    assert rc == 0 and st.true_residual <= 2e-10
    b = cont.rhs()
    assert np.linalg.norm(A.Multiply(x) - b) <= 2e-10 * np.linalg.norm(b)
    A.close()
    cont.close()
