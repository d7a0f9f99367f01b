"""The dense inverse of the AMG's coarsest level: on a mesh of at most 256 nodes
the hierarchy is that level alone, so one V-cycle is the exact solve.  Sizes
around the panel width (16 columns), the wave (64 rows) and the largest level
(1024 rows), on Newton tangents and on matrices whose diagonal blocks are zero,
which need row exchanges at every pivot."""
import numpy as np
import pytest

from tubularflowiga_amd import casegen

from test_gpu_device_api import DeviceArray, _hip, _newton_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from tubularflowiga_amd import device
    return device.Context(0)


def _dense(dm, values):
    ro, cols, _ = dm.pattern()
    n = dm.nodes
    A = np.zeros((n, 4, n, 4))
    for i in range(n):
        for k in range(ro[i], ro[i + 1]):
            A[i, :, cols[k], :] = values.reshape(-1, 4, 4)[k]
    return A.reshape(4 * n, 4 * n)


@pytest.mark.parametrize("degree,n_core,m_ring,n_axial", [(2, 1, 1, 1), (2, 1, 1, 3), (2, 1, 1, 8), (3, 1, 1, 1)])
@pytest.mark.parametrize("kind", ["tangent", "zero_diagonal"])
def test_single_level_cycle_is_the_solve(ctx, degree, n_core, m_ring, n_axial, kind):
    from tubularflowiga_amd import device
    case = casegen.make_case("tube", degree=degree, radius_mm=1.0, length_mm=2.0, n_core=n_core, m_ring=m_ring,
                             n_axial=n_axial, u_max=0.1)
    dm = device.DeviceMesh(ctx, case.mesh)
    assert dm.nodes <= 256
    hip = _hip()
    rng = np.random.default_rng(41)
    if kind == "tangent":
        values, _ = _newton_system(dm, case)
    else:
        values = rng.standard_normal((dm.nnzb, 4, 4))
        _, _, diag = dm.pattern()
        values[diag] = 0.0
        values = values.ravel()
    x = rng.standard_normal(4 * dm.nodes)
    cond = np.linalg.cond(_dense(dm, values))
    bufs = [DeviceArray(hip, np.ascontiguousarray(a)) for a in (values, dm.spmv(values, x), np.zeros_like(x))]
    amg = device.AmgPreconditioner(dm)
    print(f"coarse inverse {kind}: rows={4 * dm.nodes}", flush=True)
    try:
        amg.setup(bufs[0].ptr)
        assert len(amg.levels()) == 1
        amg.apply(bufs[1].ptr, bufs[2].ptr)
        z = bufs[2].download()
    finally:
        amg.close()
        for b in bufs:
            b.free()
        dm.close()
    # an explicit inverse by elimination with partial pivoting solves to about n eps cond(A), n <= 1024
    assert np.linalg.norm(z - x) <= 1024 * np.finfo(float).eps * cond * np.linalg.norm(x)
