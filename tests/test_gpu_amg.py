"""The automatic preconditioner on meshes without rectangle structure (cells
of a rectangle or half ring in a shuffled order): every order, a hierarchy of
one level, one that fits one workgroup, several levels in launches of their
own; stretched cells, partly prescribed faces, no memory for the hierarchy.

The residual of the returned trace is formed on the host from the exported
system.  CG stops at 1e-12 of the load; the FP64 floor of that residual, eps
||K|| ||x|| / ||b|| <= eps cond(K) ~ 2e-16 * 8 n^2 * stretch, is below 8e-11
here (n the cells along the shorter side), so the bound is 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QDEG = {1: 2, 2: 3, 3: 6, 4: 6}


def _mesh(hdg, nx, ny, ring=False, stretch=1.0):
    m = hdg.rectangle_mesh((nx, ny), jitter=0.15, seed=3 * nx + ny)
    rng = np.random.default_rng(nx * 1000 + ny)
    p = rng.permutation(len(m.cells))
    inv = np.concatenate([[0], np.argsort(p) + 1])
    faces = m.faces.copy()
    faces[:, 2:] = inv[faces[:, 2:]]
    nodes = m.nodes * [1.0, stretch]
    if ring:
        r, t = 1.0 - 0.6 * nodes[:, 0], np.pi * nodes[:, 1]
        nodes = np.stack([r * np.cos(t), r * np.sin(t)], axis=1)
        x = nodes[m.cells[:, :3] - 1]
        d = np.cross(x[:, 1] - x[:, 0], x[:, 2] - x[:, 0])
        assert (d > 0).all() or (d < 0).all()
        if d[0] < 0:
            nodes = nodes * [1.0, -1.0]
    return hdg.PolygonalMesh(nodes, m.cells[p], faces, m.facesets, m.nodesets)


def _solve(hdg, m, k, precond, dofs=None, budget=0, tau=1.0, check=True):
    with hdg.Context(0, hbm_budget=budget) as ctx:
        ctx.set_mesh(m)
        ctx.setup(k, quad_degree=QDEG[k], rtol=1e-12, tau=tau, precond=precond)
        ctx.set_source()
        d = m.boundary_dofs(k + 1) if dofs is None else dofs
        v = np.cos(np.arange(len(d)))
        ctx.set_dirichlet(d, v)
        used = ctx.memory_used()
        try:
            info = ctx.run()
        except hdg.HDGError as e:
            assert not check, e
            return None, None, used
        x = ctx.trace()
        if check:
            its = [info.iters, ctx.run().iters, ctx.run().iters]  # eager, then the captured chunks
            assert len(set(its)) == 1 and np.array_equal(ctx.trace(), x)
        K, b = ctx.get_system_scipy()
    free = np.ones(len(x), dtype=bool)
    free[d - 1] = False
    assert np.array_equal(x[~free], v[np.argsort(d)])
    lift = np.where(free, 0.0, x)
    r, b0 = (b - K @ x)[free], (b - K @ lift)[free]
    assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(b0)
    return info, x, used


@pytest.mark.parametrize("nx,ny,k,ring,stretch", [
    (1, 2, 1, False, 1.0), (5, 4, 3, False, 1.0), (8, 9, 4, True, 1.0), (23, 40, 2, True, 1.0), (44, 45, 1, False, 1.0),
    (61, 57, 3, True, 1.0), (70, 90, 4, False, 1.0), (140, 120, 2, False, 3.0), (201, 180, 1, True, 1.0)])
def test_auto_on_unstructured(hdg, nx, ny, k, ring, stretch):
    m = _mesh(hdg, nx, ny, ring, stretch)
    info, x, _ = _solve(hdg, m, k, hdg.PC_AUTO)
    ref, y, _ = _solve(hdg, m, k, hdg.PC_BLOCK_JACOBI)
    print(f"[amg] {nx}x{ny} k={k}: {info.iters} iterations, {ref.iters} without")
    assert info.iters <= ref.iters + 2 and info.iters <= 120


@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_partly_prescribed(hdg, k):
    """Prescribed: one mode of every boundary face, and of some inside."""
    m = _mesh(hdg, 30, 26)
    nt = k + 1
    bf = np.nonzero(m.faces[:, 3] == 0)[0]
    extra = np.random.default_rng(k).choice(len(m.faces), 17, replace=False)
    d = np.unique(np.concatenate([bf * nt + 1, extra * nt + 1 + k]))
    _solve(hdg, m, k, hdg.PC_AUTO, dofs=d)


def test_without_memory_for_the_hierarchy(hdg):
    """A budget that holds the block-Jacobi context exactly still solves."""
    m = _mesh(hdg, 40, 31)
    ref, y, used = _solve(hdg, m, 2, hdg.PC_BLOCK_JACOBI, check=False)
    info, x, _ = _solve(hdg, m, 2, hdg.PC_AUTO, budget=used, check=False)
    assert info.iters == ref.iters and np.array_equal(x, y)


@pytest.mark.parametrize("k,tau", [(1, 0.3), (2, 5.0), (3, 2.0), (4, 4.0), (1, 40.0)])
def test_other_tau(hdg, k, tau):
    """Solved, or refused, as block-Jacobi does."""
    m = _mesh(hdg, 21, 25, ring=True)
    ref, _, _ = _solve(hdg, m, k, hdg.PC_BLOCK_JACOBI, tau=tau, check=False)
    info, _, _ = _solve(hdg, m, k, hdg.PC_AUTO, tau=tau, check=False)
    assert (info is None) == (ref is None)
