"""Robin Hood over several workgroups (more than 8,192 unknowns): the same corrections as the
one-workgroup kernel (KRobinHood's sequence: first argmax of |b - A x|, x_i += r_i / A_ii), so
the same iterate bit for bit, the same sub-iteration count and residual; the one-workgroup
kernel is pinned against the oracle's restatement on the smaller meshes of test_gpu_parity."""
import numpy as np
import pytest

from kassiopeia_amd import geometry as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def coax12k():
    from kassiopeia_amd import kemfield as K

    ctx = K.Context(0)
    ctx.set_integrator("numeric")
    m = G.coax_mesh(nphi_in=32, nphi_out=64, nz=60, ncap_r=4, ncap_phi=40)
    assert m.n == 12160
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont)
    yield ctx, m, cont, A
    A.close()
    cont.close()
    ctx.close()


def test_grid_equals_single_workgroup(coax12k):
    from kassiopeia_amd import autotune as T

    ctx, m, cont, A = coax12k
    b = cont.rhs()
    out = {}
    for groups in (1, 0):
        T.set_knob(ctx, "robin_hood_groups", groups)
        x, st, rc = A.solve(b, method="robin_hood", tolerance=1e-9, max_iterations=12)
        print(f"Robin Hood, groups knob {groups}: {st.sub_iterations} corrections in {st.seconds:.3f} s, "
              f"residual {st.residual:.3e}", flush=True)
        out[groups] = (x, st.sub_iterations, st.residual)
    T.set_knob(ctx, "robin_hood_groups", 0)
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1] and out[0][2] == out[1][2]
    # the corrections reduce the residual (||b - A x||_inf / ||b||_inf starts at 1)
    assert out[0][2] < 0.1
    r = np.abs(b - A.Multiply(out[0][0])).max() / np.abs(b).max()
    assert r < 0.1


@pytest.mark.parametrize("n", [1, 63, 65, 256, 2048, 2049, 4097, 8191])
def test_small_matches_host_sequence(n):
    """The register kernel (up to 8,191 unknowns; 256, 512 and 1,024 threads, ragged last rows) against the same
    corrections on the host: first argmax of |b - b_iter| (all residuals alike at first), the product and the sum of
    each update fused as on the device."""
    from kassiopeia_amd import kemfield as K

    ctx = K.Context(0)
    ctx.set_integrator("numeric")
    m = G.coax_mesh(nphi_in=32, nphi_out=64, nz=60, ncap_r=4, ncap_phi=40).subset(np.arange(n))
    m.bc_value[:] = 1.0
    cont = K.KSurfaceContainer(ctx, m)
    A = K.KBoundaryIntegralMatrix(cont)
    steps = 40
    x, st, rc = A.solve(cont.rhs(), method="robin_hood", tolerance=1e-300, check_interval=steps, max_iterations=1)
    Ad = A.to_numpy()
    xr, it, b = np.zeros(n), np.zeros(n), np.ones(n)
    for _ in range(steps):
        r = b - it
        k = int(np.argmax(np.abs(r)))
        c = r[k] / Ad[k, k]
        xr[k] += c
        it += Ad[:, k] * c
    # the host rounds the product before the sum: 40 corrections of a few ulps each, on x of size one
    assert st.sub_iterations == steps
    assert np.abs(x - xr).max() <= 1e-13 * np.abs(xr).max()
    A.close()
    cont.close()
    ctx.close()
