"""A numeric rebuild that fails, because the coarsest level of the new matrix is
singular, has rebuilt all the other levels.  The handle goes on with them and
the coarsest inverse it had: the new matrix is beyond FP16 (an entry of D^-1 A
above 60000), so its cycle has to read FP32 blocks in all its steps.  A good
matrix afterwards restores the cycle of the first set-up bit for bit."""
import numpy as np
import pytest

from tubularflowiga_amd import casegen

from test_gpu_device_api import DeviceArray, _hip
from test_gpu_vcycle import _symmetric_values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,smoother", [(1, 2), (1, 0), (0, 2)])
def test_failed_update_leaves_a_usable_handle(precision, smoother):
    from tubularflowiga_amd import device
    case = casegen.make_case("tube", degree=2, radius_mm=1.0, length_mm=10.0, n_core=2, m_ring=2, n_axial=20, u_max=0.1)
    dm = device.DeviceMesh(device.Context(0), case.mesh)
    hip = _hip()
    good = _symmetric_values(dm)
    ro, cols, diag = dm.pattern()
    bad = good.reshape(-1, 4, 4).copy()
    bad[:, 3, :] = bad[:, :, 3] = 0.0       # a field without equations: zero pivots on the coarsest level
    off = next(k for k in range(ro[5], ro[6]) if k != diag[5])
    bad[off, 0, 0] = 1e9                    # and one entry of D^-1 A beyond FP16
    u = np.random.default_rng(71).standard_normal(4 * dm.nodes)
    bufs = [DeviceArray(hip, np.ascontiguousarray(a)) for a in (good, bad.ravel(), u, np.zeros_like(u))]
    dgood, dbad, du, dz = bufs
    amg = device.AmgPreconditioner(dm, precision=precision, smoother=smoother)
    try:
        amg.setup(dgood.ptr)
        print(f"failed update precision={precision} smoother={smoother} levels={amg.levels()}", flush=True)
        assert len(amg.levels()) >= 2
        amg.apply(du.ptr, dz.ptr)
        first = dz.download()
        with pytest.raises(device.TfiError, match="coarsest operator is singular"):
            amg.update(dbad.ptr)
        amg.apply(du.ptr, dz.ptr)
        assert np.all(np.isfinite(dz.download()))
        amg.update(dgood.ptr)
        amg.apply(du.ptr, dz.ptr)
        assert np.array_equal(dz.download(), first)
    finally:
        amg.close()
        for b in bufs:
            b.free()
        dm.close()
