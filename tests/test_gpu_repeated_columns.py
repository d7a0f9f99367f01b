"""Extraction rows that hold a column more than once: in the residual and the
tangent, with and without the basis table, the last entry of a column counts.
Entries put in before the true one, next to it or 8 and 40 places ahead of it,
change no bit of the results."""
import dataclasses

import numpy as np
import pytest

from tubularflowiga_amd import casegen

from meshes import split_basis

pytestmark = pytest.mark.gpu

RHO, MU = 1060.0 * (1e-3) ** 2, 3.5e-3


def _with_repeats(mesh):
    """The mesh with repeated columns in most rows, up to 90 entries a row."""
    rng = np.random.default_rng(81)
    xoff = mesh.extraction_offsets
    cols, vals = [], []
    for a in range(len(xoff) - 1):
        c = list(mesh.extraction_columns[xoff[a]:xoff[a + 1]])
        v = list(mesh.extraction_values[xoff[a]:xoff[a + 1]])
        for ahead in ((), (1,), (8,), (1, 8), (40,) * 40)[a % 5]:
            at = int(rng.integers(len(c)))
            c.insert(max(0, at - ahead + 1), c[at])
            v.insert(max(0, at - ahead + 1), float(rng.standard_normal()))
        cols.append(c)
        vals.append(v)
    return dataclasses.replace(
        mesh, extraction_offsets=np.cumsum([0] + [len(c) for c in cols]).astype(np.int32),
        extraction_columns=np.concatenate(cols).astype(np.uint8), extraction_values=np.concatenate(vals), extra={})


@pytest.mark.parametrize("degree,extra", [(2, 0), (2, 6), (3, 16)])
def test_last_entry_of_a_column_counts(degree, extra):
    from tubularflowiga_amd import device
    mesh = casegen.make_case("tube", degree=degree, radius_mm=1.0, length_mm=2.0, n_core=1, m_ring=1, n_axial=3,
                             u_max=0.1).mesh
    if extra:
        mesh = split_basis(mesh, every=2, extra=extra)
    repeats = _with_repeats(mesh)
    for a in range(len(mesh.connectivity)):
        row = dict(zip(repeats.extraction_columns[repeats.extraction_offsets[a]:repeats.extraction_offsets[a + 1]],
                       repeats.extraction_values[repeats.extraction_offsets[a]:repeats.extraction_offsets[a + 1]]))
        lo, hi = mesh.extraction_offsets[a], mesh.extraction_offsets[a + 1]
        assert row == dict(zip(mesh.extraction_columns[lo:hi], mesh.extraction_values[lo:hi]))
    print(f"repeated columns nen={mesh.maximum_basis}: longest row {np.diff(repeats.extraction_offsets).max()}", flush=True)
    ctx = device.Context(0)
    state = np.random.default_rng(82).standard_normal(4 * mesh.nodes)
    got = []
    for m in (mesh, repeats):
        dm = device.DeviceMesh(ctx, m)
        try:
            for table in (1, 0):
                dm.basis_table(table)
                got.append((*dm.assemble(state, 0.5 * state, RHO, MU, 1e-3),
                            dm.assemble(state, 0.5 * state, RHO, MU, 1e-3, jacobian=False)[1]))
        finally:
            dm.close()
    for plain, repeated in ((got[0], got[2]), (got[1], got[3])):
        for x, y in zip(plain, repeated):
            assert np.array_equal(x, y)
