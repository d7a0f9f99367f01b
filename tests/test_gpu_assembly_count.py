"""The arithmetic that the timers count for an assembly: a residual alone does not
evaluate the basis, with the basis table or without; a tangent does without."""
import numpy as np
import pytest

from tubularflowiga_amd import casegen

pytestmark = pytest.mark.gpu


def test_counted_flops_follow_the_work():
    from tubularflowiga_amd import device
    mesh = casegen.make_case("tube", degree=2, radius_mm=1.0, length_mm=2.0, n_core=1, m_ring=1, n_axial=2, u_max=0.1).mesh
    ctx = device.Context(0)
    dm = device.DeviceMesh(ctx, mesh)
    state = np.random.default_rng(3).standard_normal(4 * mesh.nodes)
    counted = {}
    try:
        for table in (1, 0):
            dm.basis_table(table)
            for jacobian in (False, True):
                ctx.timers(enable=True, reset=True)
                dm.assemble(state, state, 1.0, 0.1, 1e-3, jacobian=jacobian)
                t = ctx.timers(enable=False)
                counted[table, jacobian] = t["assembly_flops"] if jacobian else t["residual_flops"]
                assert counted[table, jacobian] == dm.assembly_flops("exact", jacobian)
    finally:
        dm.close()
    entries = float(np.diff(mesh.element_offsets).sum())
    assert counted[0, False] == counted[1, False] == 64.0 * (82.0 * entries + 300.0 * mesh.elements)
    assert counted[0, True] - counted[1, True] == 64.0 * 698.0 * entries
