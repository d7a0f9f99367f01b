"""The residual-only assembly and the node sums against the CPU oracle at the
element sizes where the kernel's loops change: 27 basis functions, meshes
mixing 27 with 33, 64 (every lane a basis function) and meshes mixing 64 with
65 and 80; five to fifteen elements; transient and steady."""
import dataclasses

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


def _mesh(name):
    degree, n_axial, extra = {"nen27": (2, 1, 0), "nen33": (2, 3, 6), "nen64": (3, 1, 0), "nen65": (3, 2, 1),
                              "nen80": (3, 3, 16)}[name]
    m = casegen.make_case("tube", degree=degree, radius_mm=1.0, length_mm=2.0, n_core=1, m_ring=1, n_axial=n_axial,
                          u_max=0.1).mesh
    return split_basis(m, every=2, extra=extra) if extra else m


@pytest.mark.parametrize("dt", [1e-3, 0.0])
@pytest.mark.parametrize("name", ["nen27", "nen33", "nen64", "nen65", "nen80"])
def test_residual_matches_oracle(ctx, name, dt):
    from tubularflowiga_amd import device
    mesh = _mesh(name)
    print(f"residual {name}: elements={mesh.elements} nodes={mesh.nodes} nen={mesh.maximum_basis} dt={dt}", flush=True)
    rng = np.random.default_rng(21)
    state = np.concatenate([50.0 * rng.standard_normal((mesh.nodes, 3)), 10.0 * rng.standard_normal((mesh.nodes, 1))],
                           axis=1).ravel()
    previous = 0.5 * state[::-1].copy()
    dm = device.DeviceMesh(ctx, mesh)
    try:
        _, got = dm.assemble(state, previous, RHO, MU, dt, jacobian=False)
        _, again = dm.assemble(state, previous, RHO, MU, dt, jacobian=False)
    finally:
        dm.close()
    _, want = O.ns_assemble(mesh, O.block_pattern(mesh), state, previous, RHO, MU, dt, "exact")
    # FP64 sums of at most 64 nen terms per point and 64 points in another order:
    # measured below 2e-15 of the largest entry; the bound is that of the full assembly's test
    assert np.max(np.abs(got - want)) <= 1e-11 * np.max(np.abs(want))
    assert np.array_equal(got, again)


@pytest.mark.parametrize("name", ["nen27", "nen33"])
def test_long_extraction_rows(ctx, name):
    """Rows of 31, 32, 33 and 64 stored entries (a lane holds the first four of its
    eighth of a row and walks the rest): zeros stored beside the entries of the
    same operator leave the residual as it is."""
    from tubularflowiga_amd import device
    mesh = _mesh(name)
    xoff = mesh.extraction_offsets
    cols, vals = [], []
    for i in range(len(xoff) - 1):
        own = mesh.extraction_columns[xoff[i]:xoff[i + 1]]
        rest = np.setdiff1d(np.arange(64), own)
        keep = np.sort(np.concatenate([own, rest[:(31, 32, 33, 64)[i % 4] - len(own)]]))
        row = np.zeros(64)
        row[own] = mesh.extraction_values[xoff[i]:xoff[i + 1]]
        cols.append(keep)
        vals.append(row[keep])
    long = dataclasses.replace(
        mesh, extraction_offsets=np.cumsum([0] + [len(c) for c in cols]).astype(np.int32),
        extraction_columns=np.concatenate(cols).astype(np.uint8), extraction_values=np.concatenate(vals), extra={})
    rng = np.random.default_rng(22)
    state = rng.standard_normal(4 * mesh.nodes)
    got = []
    for m in (mesh, long):
        dm = device.DeviceMesh(ctx, m)
        try:
            got.append(dm.assemble(state, 0.5 * state, RHO, MU, 1e-3, jacobian=False)[1])
        finally:
            dm.close()
    # the same sums with zeros between their terms; 1e-13 leaves room for their order
    assert np.max(np.abs(got[1] - got[0])) <= 1e-13 * np.max(np.abs(got[0]))
