"""The matrix-core tangent against the CPU oracle where its tiles and loops
change: 27 / 28 basis functions (the last trial function of a wave idle or
not), 32, 33 (two and three test tiles), 48, 49, 64, 65 and 80, meshes mixing
these with smaller elements, with and without the basis table, and a mesh whose
element blocks are too large to stage, so that it is assembled by colour."""
import numpy as np
import pytest

from oracle import oracle as O
from tubularflowiga_amd import casegen

from meshes import split_basis

pytestmark = pytest.mark.gpu

RHO, MU = 1060.0 * (1e-3) ** 2, 3.5e-3


@pytest.fixture(scope="module")
def ctx():
    from tubularflowiga_amd import device
    return device.Context(0)


def _tube(degree, n_core, m_ring, n_axial):
    return casegen.make_case("tube", degree=degree, radius_mm=1.0, length_mm=2.0, n_core=n_core, m_ring=m_ring,
                             n_axial=n_axial, u_max=0.1).mesh


def _mesh(nen):
    degree, base = (2, 27) if nen <= 54 else (3, 64)
    m = _tube(degree, 1, 1, 3)
    return split_basis(m, every=2, extra=nen - base) if nen > base else m


def _state(nodes, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([50.0 * rng.standard_normal((nodes, 3)), 10.0 * rng.standard_normal((nodes, 1))],
                          axis=1).ravel()


def _check(dm, mesh, dt, tangent):
    state, previous = _state(mesh.nodes, 31), _state(mesh.nodes, 32)
    jac, res = dm.assemble(state, previous, RHO, MU, dt, tangent=tangent)
    again, _ = dm.assemble(state, previous, RHO, MU, dt, tangent=tangent)
    ojac, ores = O.ns_assemble(mesh, O.block_pattern(mesh), state, previous, RHO, MU, dt, tangent)
    # FP64 sums in another order: measured below 1e-14 of the largest entry; the
    # bound is that of the assembly tests at the usual element sizes
    assert np.max(np.abs(jac - ojac)) <= 1e-11 * np.max(np.abs(ojac))
    assert np.max(np.abs(res - ores)) <= 1e-11 * np.max(np.abs(ores))
    assert np.array_equal(jac, again)


@pytest.mark.parametrize("table", [1, 0])
@pytest.mark.parametrize("nen", [27, 28, 32, 33, 48, 49, 64, 65, 80])
def test_tangent_matches_oracle(ctx, nen, table):
    from tubularflowiga_amd import device
    mesh = _mesh(nen)
    assert mesh.maximum_basis == nen
    print(f"tangent nen={nen} table={table}: elements={mesh.elements} nodes={mesh.nodes}", flush=True)
    dm = device.DeviceMesh(ctx, mesh)
    try:
        dm.basis_table(table)
        for dt in (1e-3, 0.0):
            for tangent in ("exact", "legacy"):
                _check(dm, mesh, dt, tangent)
    finally:
        dm.close()


@pytest.mark.parametrize("nen", [27, 64])
def test_wide_workgroups_match_oracle(ctx, nen):
    """Enough elements for the widest workgroups (all trial functions of 27, 16 of 64)."""
    from tubularflowiga_amd import device
    mesh = _tube(2, 3, 3, 14) if nen == 27 else _tube(3, 2, 2, 8)
    print(f"tangent nen={nen}: elements={mesh.elements} nodes={mesh.nodes}", flush=True)
    dm = device.DeviceMesh(ctx, mesh)
    try:
        _check(dm, mesh, 1e-3, "exact")
    finally:
        dm.close()


def test_assembly_by_colour_matches_oracle(ctx):
    from tubularflowiga_amd import device
    mesh = _tube(2, 6, 6, 260)
    assert 128 * 27 * 27 * mesh.elements > 4 << 30
    print(f"tangent by colour: elements={mesh.elements} nodes={mesh.nodes}", flush=True)
    dm = device.DeviceMesh(ctx, mesh)
    try:
        _check(dm, mesh, 1e-3, "exact")
    finally:
        dm.close()
