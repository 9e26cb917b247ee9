"""Meshes numbered like rectangle_mesh whose faces are not the grid's: cut open
along an axis edge, along a diagonal, along a line of edges, with the sides
joined, with two edges' faces exchanged between the joined sides.  Cells and
nodes alone do not tell them from the grid; every preconditioner and precision
that takes the numbering has to solve the system of the mesh's own faces.

The residual of the returned trace is formed on the host from the exported
system (poisson2D_HDG.jl:176-195).  CG stops at 1e-12 of the load; the FP64 floor
of that residual, eps cond(K) ~ 2e-16 * 8 n^2, is below 1e-11 for the 40 cells
per side here, so the bound is 5e-11.  Both faces of a cut carry values of their
own: the system's size says so, and the prescribed one of a cut is met while
the other stays free."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _cut(m, which):
    """Face f of two cells becomes two faces of one cell each."""
    cells, faces = m.cells.copy(), m.faces.copy()
    for f in which:
        c = faces[f, 3]
        faces[f, 3] = 0
        faces = np.vstack([faces, [faces[f, 0], faces[f, 1], c, 0]])
        cells[c - 1, 3:][cells[c - 1, 3:] == f + 1] = len(faces)
    return cells, faces


def _join(m, nx, ny, swap=False):
    """The left and the right side's faces become one, row by row."""
    cells, faces = m.cells.copy(), m.faces.copy()
    rows = np.arange(ny)
    left = cells[2 * rows * nx, 4] - 1
    right = cells[2 * (rows * nx + nx - 1) + 1, 5] - 1
    if swap:
        right = right.copy()
        right[[0, 1]] = right[[1, 0]]
    for a, b in zip(left, right):
        c = faces[b, 2]
        faces[a, 3] = c
        cells[c - 1, 3:][cells[c - 1, 3:] == b + 1] = a + 1
    keep = np.setdiff1d(np.arange(len(faces)), right)
    new = np.zeros(len(faces) + 1, dtype=np.int64)
    new[keep + 1] = np.arange(1, len(keep) + 1)
    cells[:, 3:] = new[cells[:, 3:]]
    return cells, faces[keep]


def _mesh(hdg, nx, ny, kind):
    m = hdg.rectangle_mesh((nx, ny), jitter=0.2, seed=nx + ny)
    f = m.faces
    diag = np.nonzero((f[:, 3] > 0) & ((f[:, 2] - 1) // 2 == (f[:, 3] - 1) // 2))[0]
    axis = np.setdiff1d(np.nonzero(f[:, 3] > 0)[0], diag)
    nodes = m.nodes.copy()
    if kind == "axis":
        cells, faces = _cut(m, axis[len(axis) // 2: len(axis) // 2 + 1])
    elif kind == "diagonal":
        cells, faces = _cut(m, diag[len(diag) // 2: len(diag) // 2 + 1])
    elif kind == "line":
        row = {i + (ny // 2) * (nx + 1) + 1 for i in range(nx + 1)}
        line = [a for a in axis if f[a, 0] in row and f[a, 1] in row]
        assert len(line) == nx
        cells, faces = _cut(m, line[: nx - 1])
    else:
        # the joined sides carry the same heights
        g = np.arange(ny + 1) * (nx + 1)
        nodes[g + nx, 1] = nodes[g, 1]
        cells, faces = _join(m, nx, ny, kind == "swapped")
    return hdg.PolygonalMesh(nodes, cells, faces, {}, {})


def _solve(hdg, m, k, precond, precision):
    nt = k + 1
    bf = np.nonzero(m.faces[:, 3] == 0)[0]
    # every other face of one cell is prescribed: one side of some cuts, none of others
    d = (bf[::2, None] * nt + np.arange(1, nt + 1)).ravel()
    v = np.cos(np.arange(len(d)))
    with hdg.Context(0) as ctx:
        ctx.set_mesh(m)
        ctx.setup(k, quad_degree=QD[k], rtol=1e-12, precond=precond, precision=precision)
        ctx.set_source()
        ctx.set_dirichlet(d, v)
        info = ctx.run()
        x = ctx.trace()
        assert ctx.run().iters == info.iters and np.array_equal(ctx.trace(), x)
        K, b = ctx.get_system_scipy()
    assert len(x) == len(m.faces) * nt == len(b)
    free = np.ones(len(x), dtype=bool)
    free[d - 1] = False
    assert np.array_equal(x[~free], v)
    lift = np.where(free, 0.0, x)
    res = np.linalg.norm((b - K @ x)[free]) / np.linalg.norm((b - K @ lift)[free])
    return info, res


@pytest.mark.parametrize("kind", ["axis", "diagonal", "line", "joined", "swapped"])
@pytest.mark.parametrize("nx,ny,k", [(2, 3, 1), (3, 2, 4), (12, 9, 2), (40, 33, 1), (31, 40, 3)])
def test_other_faces(hdg, nx, ny, k, kind):
    m = _mesh(hdg, nx, ny, kind)
    ref, res = _solve(hdg, m, k, hdg.PC_BLOCK_JACOBI, 0)
    assert res < 5e-11
    for precond, precision in ((hdg.PC_AUTO, 0), (hdg.PC_MULTIGRID, 0), (hdg.PC_AUTO, hdg.HDG_MIXED)):
        print(f"[faces] {nx}x{ny} k={k} {kind} precond={precond} precision={precision}", flush=True)
        info, res = _solve(hdg, m, k, precond, precision)
        print(f"    {info.iters} iterations ({ref.iters} of block-Jacobi), residual {res:.1e}, device {info.true_relres:.1e}",
              flush=True)
        assert res < 5e-11 and info.true_relres < 5e-11
        # the V-cycle still preconditions: a hierarchy over the mesh's own vertices
        assert info.iters <= max(ref.iters // 2, 60) or kind == "swapped"


@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_grid_faces_in_another_order(hdg, k):
    """The grid's own faces under other ids are the grid: the same solution in
    the same number of iterations."""
    m = hdg.rectangle_mesh((17, 12), jitter=0.2, seed=k)
    p = np.random.default_rng(k).permutation(len(m.faces))  # new face i is old face p[i]
    cells = m.cells.copy()
    cells[:, 3:] = (np.argsort(p) + 1)[cells[:, 3:] - 1]
    faces = m.faces[p]
    two = faces[:, 3] > 0
    faces[two, 2:] = faces[two][:, [3, 2]]
    q = hdg.PolygonalMesh(m.nodes, cells, faces, {}, {})
    out = []
    for mesh in (m, q):
        with hdg.Context(0) as ctx:
            ctx.set_mesh(mesh)
            ctx.setup(k, quad_degree=QD[k], rtol=1e-12, precond=hdg.PC_MULTIGRID)
            ctx.set_source()
            ctx.set_dirichlet_boundary(0.0)
            out.append((ctx.run().iters, ctx.trace().reshape(-1, k + 1)))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1][p], out[1][1])
