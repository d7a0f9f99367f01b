"""The tangent added to the Jacobian element colour by element colour, and the
one summed from staged element blocks: both leave in a block the sum of its
elements' contributions in the order of their colours, bit for bit, so which of
them a mesh takes (its size and the free memory decide) changes no result.  The
contributions come from meshes of a single element.  By colour the blocks are
added by atomics in the GPU's own memory, and by loads and stores elsewhere: in
pinned host memory the same bits come out."""
import ctypes
import dataclasses

import numpy as np
import pytest

from tubularflowiga_amd import casegen

from test_gpu_device_api import DeviceArray, _hip

pytestmark = pytest.mark.gpu

RHO, MU, DT = 1060.0 * (1e-3) ** 2, 3.5e-3, 1e-3


@pytest.fixture(scope="module")
def ctx():
    from tubularflowiga_amd import device
    return device.Context(0)


def _tube(n_core, m_ring, n_axial, degree=2):
    return casegen.make_case("tube", degree=degree, radius_mm=1.0, length_mm=2.0, n_core=n_core, m_ring=m_ring,
                             n_axial=n_axial, u_max=0.1).mesh


def _state(nodes):
    return np.random.default_rng(91).standard_normal(4 * nodes)


def _element_blocks(ctx, mesh, e, state, previous):
    """[nen, nen, 16] contributions of element e, from a mesh of that element alone."""
    from tubularflowiga_amd import device
    b0, b1 = mesh.element_offsets[e], mesh.element_offsets[e + 1]
    x0, x1 = mesh.extraction_offsets[b0], mesh.extraction_offsets[b1]
    nodes = mesh.connectivity[b0:b1]
    nen = len(nodes)
    single = dataclasses.replace(
        mesh, nodes=nen, element_offsets=np.array([0, nen], np.int32), connectivity=np.arange(nen, dtype=np.int32),
        extraction_offsets=(mesh.extraction_offsets[b0:b1 + 1] - x0).astype(np.int32),
        extraction_columns=mesh.extraction_columns[x0:x1], extraction_values=mesh.extraction_values[x0:x1],
        bezier_points=mesh.bezier_points.reshape(-1, 192)[e], extra={})
    dm = device.DeviceMesh(ctx, single)
    try:
        jac, _ = dm.assemble(state.reshape(-1, 4)[nodes].ravel(), previous.reshape(-1, 4)[nodes].ravel(), RHO, MU, DT)
    finally:
        dm.close()
    return jac.reshape(nen, nen, 16)


def _check_rows(ctx, dm, mesh, jac, rows, state, previous):
    ro, cols, _ = dm.pattern()
    colors = dm.colors()
    jac = jac.reshape(-1, 16)
    owner = np.repeat(np.arange(mesh.elements), np.diff(mesh.element_offsets))
    for i in rows:
        elements = np.unique(owner[mesh.connectivity == i])
        want = np.zeros((ro[i + 1] - ro[i], 16))
        for e in elements[np.argsort(colors[elements], kind="stable")]:
            nodes = mesh.connectivity[mesh.element_offsets[e]:mesh.element_offsets[e + 1]]
            blocks = _element_blocks(ctx, mesh, e, state, previous)[np.flatnonzero(nodes == i)[0]]
            want[np.searchsorted(cols[ro[i]:ro[i + 1]], nodes)] += blocks
        assert np.array_equal(jac[ro[i]:ro[i + 1]], want), f"row {i}"


@pytest.mark.parametrize("degree", [2, 3])
def test_staged_sums_in_colour_order(ctx, degree):
    from tubularflowiga_amd import device
    mesh = _tube(1, 1, 4, degree)
    state, previous = _state(mesh.nodes), 0.5 * _state(mesh.nodes)
    dm = device.DeviceMesh(ctx, mesh)
    try:
        jac, _ = dm.assemble(state, previous, RHO, MU, DT)
        print(f"staged degree={degree} elements={mesh.elements}", flush=True)
        _check_rows(ctx, dm, mesh, jac, range(0, mesh.nodes, 7), state, previous)
    finally:
        dm.close()


def test_by_colour_in_device_and_pinned_memory(ctx):
    from tubularflowiga_amd import device
    mesh = _tube(6, 6, 260)
    assert 128 * 27 * 27 * mesh.elements > 4 << 30      # too large to stage
    state, previous = _state(mesh.nodes), 0.5 * _state(mesh.nodes)
    hip = _hip()
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    dm = device.DeviceMesh(ctx, mesh)
    pinned = ctypes.c_void_p()
    bufs = []
    try:
        jac, _ = dm.assemble(state, previous, RHO, MU, DT)
        print(f"by colour elements={mesh.elements} blocks={dm.nnzb}", flush=True)
        _check_rows(ctx, dm, mesh, jac, np.random.default_rng(92).integers(0, mesh.nodes, 4), state, previous)
        assert hip.hipHostMalloc(ctypes.byref(pinned), jac.nbytes, 0) == 0
        bufs = [DeviceArray(hip, a) for a in (state, previous, np.zeros_like(state))]
        dm.ctx.check(dm.lib.tfi_ns_assemble_device(dm.handle, bufs[0].ptr, bufs[1].ptr, RHO, MU, DT, pinned,
                                                   bufs[2].ptr, 1))
        got = np.ctypeslib.as_array(ctypes.cast(pinned, ctypes.POINTER(ctypes.c_double)), (16 * dm.nnzb,))
        assert np.array_equal(got, jac.ravel())
    finally:
        for b in bufs:
            b.free()
        if pinned:
            hip.hipHostFree(pinned)
        dm.close()
