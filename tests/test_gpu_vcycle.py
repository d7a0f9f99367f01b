"""The V-cycle's smoothing around the coarse correction: for a symmetric
positive definite matrix, as many steps of the same D^-1 A polynomial before and
after a Galerkin correction make the cycle a symmetric operator, (M^-1 u, v) =
(u, M^-1 v); a step after the correction that missed a term of the corrected
residual would not.  Two levels, Chebyshev and Jacobi smoothing, FP64
and FP32 / FP16, and the result written over the input."""
import numpy as np
import pytest

from tubularflowiga_amd import casegen

from test_gpu_device_api import DeviceArray, _hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from tubularflowiga_amd import device
    return device.Context(0)


def _symmetric_values(dm):
    """A weighted graph Laplacian with 4x4 SPD couplings, plus a mass term."""
    ro, cols, diag = dm.pattern()
    rng = np.random.default_rng(61)
    rows = np.repeat(np.arange(dm.nodes), np.diff(ro))
    slot = {(int(i), int(j)): k for k, (i, j) in enumerate(zip(rows, cols))}
    values = np.zeros((dm.nnzb, 4, 4))
    for k, (i, j) in enumerate(zip(rows, cols)):
        if i < j:
            B = rng.standard_normal((4, 4))
            W = (0.1 * B @ B.T + np.eye(4)) * rng.uniform(0.2, 1.0)
            values[k] = -W
            values[slot[(int(j), int(i))]] = -W
            values[diag[i]] += W
            values[diag[j]] += W
    values[diag] += 0.05 * np.eye(4)
    return values.ravel()


@pytest.mark.parametrize("mesh", [(1, 1, 16), (2, 2, 60)])
@pytest.mark.parametrize("precision,smoother", [(0, 2), (0, 0), (1, 2), (1, 0)])
def test_cycle_is_symmetric(ctx, mesh, precision, smoother):
    from tubularflowiga_amd import device
    n_core, m_ring, n_axial = mesh
    case = casegen.make_case("tube", degree=2, radius_mm=1.0, length_mm=10.0, n_core=n_core, m_ring=m_ring,
                             n_axial=n_axial, u_max=0.1)
    dm = device.DeviceMesh(ctx, case.mesh)
    hip = _hip()
    values = _symmetric_values(dm)
    rng = np.random.default_rng(62)
    u, v = rng.standard_normal((2, 4 * dm.nodes))
    bufs = [DeviceArray(hip, a) for a in (values, u, v, np.zeros_like(u))]
    da, du, dv, dz = bufs
    amg = device.AmgPreconditioner(dm, precision=precision, smoother=smoother)
    try:
        amg.setup(da.ptr)
        print(f"v-cycle nodes={dm.nodes} precision={precision} smoother={smoother} levels={amg.levels()}", flush=True)
        assert len(amg.levels()) >= 2
        amg.apply(du.ptr, dz.ptr)
        mu = dz.download()
        amg.apply(dv.ptr, dz.ptr)
        mv = dz.download()
        amg.apply(dv.ptr, dv.ptr)
        assert np.array_equal(dv.download(), mv)
        skew = abs(mu @ v - u @ mv) / (np.linalg.norm(mu) * np.linalg.norm(v))
        # FP64: rounding of sums of 4 nodes terms; FP32 vectors and inverses: 1e-6 of them; S in FP16 is D^-1 A
        # with relative errors of 2^-11 per entry, averaged over a row
        assert skew <= {(0, 0): 1e-12, (0, 2): 1e-12, (1, 0): 1e-5, (1, 2): 2.0 ** -11}[(precision, smoother)]
        # and it is a contraction for the matrix: ||u - M^-1 A u||_A < ||u||_A
        Au = dm.spmv(values, u)
        du.upload(Au)
        amg.apply(du.ptr, dz.ptr)
        e = u - dz.download()
        assert e @ dm.spmv(values, e) < 0.9 * (u @ Au)
    finally:
        amg.close()
        for b in bufs:
            b.free()
        dm.close()
