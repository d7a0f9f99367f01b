"""The product of the configured transport's F x F block matrix, for every
supported number of fields (64 lanes are not a multiple of 3, 5, 6 or 7 rows):
a step solved with it satisfies the assembled system as a direct solver on the
host does.  Rows of the matrix hold from 8 blocks (a corner of the mesh) up."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg

from oracle import solve as S
from tubularflowiga_amd import casegen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mesh():
    from tubularflowiga_amd import device
    case = casegen.make_case("tube", degree=2, radius_mm=1.0, length_mm=10.0, n_core=1, m_ring=1, n_axial=9, u_max=0.1)
    return case, device.DeviceMesh(device.Context(0), case.mesh)


@pytest.mark.parametrize("fields", range(1, 9))
def test_step_solves_the_assembled_system(mesh, fields):
    from tubularflowiga_amd import device
    case, dm = mesh
    terms = []
    for f in range(fields):
        terms += [(S.TIME_DERIVATIVE, f, f, 1.0 + 0.1 * f), (S.DIFFUSION, f, f, 0.02 + 0.01 * f),
                  (S.LINEAR_COUPLING, f, (f + 1) % fields, 0.3), (S.LINEAR_COUPLING, f, (f + 3) % fields, -0.2),
                  (S.VOLUME_SOURCE, f, f, 0.1)]
    zeros = np.zeros((dm.nodes, fields))
    tr = device.ConfiguredTransport(dm, fields, terms, [S.SUPG_NONE] * fields, [0.0] * fields, 1e-2,
                                    np.zeros((dm.nodes, 3)), zeros.astype(np.int32))
    old = np.random.default_rng(fields).standard_normal((dm.nodes, fields))
    try:
        print(f"solve product fields={fields} nodes={dm.nodes}", flush=True)
        tr.set_boundary(zeros)
        tr.set_state(old)
        L, P, source, _ = tr.matrices()
        tr.step(zero_guess=True, rtol=1e-13)
        got = tr.state()
    finally:
        tr.close()
    ro, cols, _ = dm.pattern()
    shape = (fields * dm.nodes,) * 2
    left = sp.bsr_matrix((L, cols, ro), shape=shape)
    right = sp.bsr_matrix((P, cols, ro), shape=shape) @ old.ravel() + source.ravel()
    want = scipy.sparse.linalg.spsolve(left.tocsc(), right).reshape(-1, fields)
    # the step's rows are scaled to unit diagonal blocks and its residual is 1e-13 of
    # the right-hand side: the error is that times the condition, below 1e3 here
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"fields={fields}: rel L2 = {rel:.2e}", flush=True)
    assert rel <= 1e-10
