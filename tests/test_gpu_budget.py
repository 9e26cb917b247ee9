"""Exports under a budget that just holds a solve: the assembled matrix takes
the reduced system's place (or the aggregation hierarchy's) and gives it back
to the next solve, with the same bits as without a budget."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _setup(ctx, m, k, precision=0):
    ctx.set_mesh(m)
    ctx.setup(k, quad_degree=QD[k], precision=precision, rtol=1e-12)
    ctx.set_source()
    d = m.boundary_dofs(k + 1)
    ctx.set_dirichlet(d, np.cos(np.arange(len(d))))


def _flow(ctx):
    out = []
    for _ in range(2):  # twice: the second round starts from the export's state
        for _ in range(3):  # eager, then the captured chunks
            ctx.run()
            out.append(ctx.trace())
        K, b = ctx.get_system_scipy()
        out += [K.data, b]
        ctx.solve()
        out.append(ctx.trace())
    out += [np.asarray(a) for a in ctx.get_applied_system()]
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_exports_in_the_place_of_the_solver(hdg, k, precision):
    print(f"[budget] k={k} precision={precision}", flush=True)
    m = hdg.rectangle_mesh((40, 33), jitter=0.2, seed=k)
    with hdg.Context(0) as ctx:
        _setup(ctx, m, k, precision)
        ctx.run()
        used = ctx.memory_used()
        ref = _flow(ctx)
    nt, n = k + 1, len(ref[0])
    # beside the solve: one face-ELL and rhs, the working copy of the last export
    with hdg.Context(0, hbm_budget=used + 8 * (5 * nt * n + n + 1025)) as ctx:
        _setup(ctx, m, k, precision)
        got = _flow(ctx)
        assert ctx.memory_used() <= used + 8 * (5 * nt * n + n + 1025)
    for a, b in zip(ref, got):
        assert np.array_equal(a, b)


def test_export_in_the_place_of_the_hierarchy(hdg):
    m = hdg.rectangle_mesh((40, 31), jitter=0.15, seed=7)
    p = np.random.default_rng(5).permutation(len(m.cells))
    inv = np.concatenate([[0], np.argsort(p) + 1])
    faces = m.faces.copy()
    faces[:, 2:] = inv[faces[:, 2:]]
    m = hdg.PolygonalMesh(m.nodes, m.cells[p], faces, m.facesets, m.nodesets)
    k = 2
    with hdg.Context(0) as ctx:
        _setup(ctx, m, k)
        base = ctx.memory_used()
        ctx.run()
        used = ctx.memory_used()
        ref = _flow(ctx)
    nt, n = k + 1, len(ref[0])
    with hdg.Context(0, hbm_budget=max(used, base + 8 * (5 * nt * n + n + 1025))) as ctx:
        _setup(ctx, m, k)
        ctx.run()
        assert ctx.memory_used() > base  # the hierarchy was made
        got = _flow(ctx)
    for a, b in zip(ref, got):
        assert np.array_equal(a, b)
