"""The exports that write the caller's layout on the device and leave through
pinned chunks: one cell, sizes below, at and beyond one chunk (4 MB) and of
ragged ends, every order.  Everything is a copy, so all comparisons are exact;
only K against the sum of its cells' blocks allows for the order of two
additions and for the symmetric storage (1e-12 of the largest entry)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(hdg, nx, ny, k, annulus=False):
    m = hdg.rectangle_mesh((nx, ny), jitter=0.2, seed=nx + ny)
    if annulus:  # the same cells in another order: a mesh without structure
        p = np.random.default_rng(nx).permutation(len(m.cells))
        cells, faces = m.cells[p].copy(), m.faces.copy()
        inv = np.empty(len(p) + 1, dtype=np.int64)
        inv[0], inv[p + 1] = 0, np.arange(1, len(p) + 1)
        faces[:, 2:] = inv[faces[:, 2:]]
        m = hdg.PolygonalMesh(m.nodes, cells, faces, m.facesets, m.nodesets)
    ctx = hdg.Context(0)
    ctx.set_mesh(m)
    ctx.setup(k, quad_degree={1: 2, 2: 3, 3: 6, 4: 6}[k])
    ctx.set_source()
    ctx.assemble_condense()
    return m, ctx


@pytest.mark.parametrize("nx,ny,k,annulus", [(1, 1, 1, False), (3, 2, 4, False), (17, 31, 2, True), (64, 61, 3, False),
                                             (90, 83, 4, True), (150, 171, 1, False), (140, 133, 2, False)])
def test_exports(hdg, nx, ny, k, annulus):
    m, ctx = _case(hdg, nx, ny, k, annulus)
    with ctx:
        s = ctx.sizes
        x = np.random.default_rng(k).standard_normal(s.n_dofs)
        ctx.set_trace(x)
        assert np.array_equal(ctx.trace(), x)
        q, u, uc = ctx.recover()
        idx = (m.cells[:, 3:] - 1)[:, :, None] * s.nt + np.arange(s.nt)
        assert np.array_equal(uc, x[idx].transpose(0, 2, 1))
        rows = np.full((s.n_cells, s.nq), np.nan), np.full((s.n_cells, s.nu), np.nan), np.full_like(uc, np.nan, order="C")
        ctx.recover_into(*rows)
        for a, b in zip(rows, (q, u, uc)):
            assert np.array_equal(a, b)
        other = tuple(np.asfortranarray(np.zeros_like(a)) for a in rows)  # the general path
        ctx.recover_into(*other)
        for a, b in zip(rows, other):
            assert np.array_equal(a, b)
        Ke, be = ctx.get_local_ops()
        dof = np.einsum("cij,cj->ci", Ke, x[idx.reshape(s.n_cells, -1)]) + be
        assert np.abs(np.hstack([q, u]) - dof).max() <= 1e-11 * np.abs(dof).max()
        K, rhs = ctx.get_system_scipy()
        colptr, rowval, nzval, rhs2 = ctx.get_system()
        assert K.indices.dtype == np.int32 and K.nnz == s.nnz
        assert np.array_equal(K.indptr, colptr - 1) and np.array_equal(K.indices, rowval - 1)
        assert np.array_equal(K.data, nzval) and np.array_equal(rhs, rhs2)
        At, bt = ctx.get_condensed()
        import scipy.sparse as sp
        ci = idx.reshape(s.n_cells, -1)
        ref = sp.csc_matrix((At.ravel(), (np.repeat(ci, s.ntr, axis=1).ravel(), np.tile(ci, (1, s.ntr)).ravel())),
                            shape=K.shape)
        assert K.has_sorted_indices and abs(K - ref).max() <= 1e-12 * abs(ref).max()
        b = np.zeros(s.n_dofs)
        np.add.at(b, ci.ravel(), bt.ravel())
        assert np.abs(b - rhs).max() <= 1e-12 * np.abs(b).max()
