"""Stretched cells without rectangle structure: at odd orders the automatic
preconditioner is block-Jacobi, bit for bit, where the mesh is fewer layers
across than a multiple of the cells' aspect, and the V-cycle beyond; at even
orders the V-cycle throughout; also after a set-up of another order has left its
hierarchy there.  Mixed shapes go by the quarter of the cells that is the most
stretched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _mesh(hdg, n, scale, part=1.0):
    m = hdg.rectangle_mesh((n, n), jitter=0.15 if part == 1.0 else 0.0, seed=n)  # (rows of two scales would fold)
    p = np.random.default_rng(n).permutation(len(m.cells))
    faces = m.faces.copy()
    faces[:, 2:] = np.concatenate([[0], np.argsort(p) + 1])[faces[:, 2:]]
    y = m.nodes[:, 1]
    # the rows up to `part` stretched, the others as they were
    y = np.where(y <= part, scale * y, scale * part + (y - part))
    return hdg.PolygonalMesh(np.stack([m.nodes[:, 0], y], axis=1), m.cells[p], faces, m.facesets, m.nodesets)


def _run(ctx, hdg, k, precond):
    ctx.setup(k, quad_degree=QD[k], precond=precond)
    ctx.set_source()
    ctx.set_dirichlet_boundary(0.0)
    return ctx.run().iters, ctx.trace()


@pytest.mark.parametrize("n,k,scale,part,jacobi", [
    (12, 1, 20.0, 1.0, True), (12, 1, 0.05, 1.0, True), (12, 1, 5.0, 1.0, False), (40, 1, 20.0, 1.0, False),
    (40, 1, 100.0, 1.0, True), (12, 3, 14.0, 1.0, False), (12, 3, 50.0, 1.0, True), (12, 2, 100.0, 1.0, False),
    (12, 4, 100.0, 1.0, False), (12, 1, 100.0, 0.5, True), (12, 1, 100.0, 0.1, False)])
def test_choice(hdg, n, k, scale, part, jacobi):
    m = _mesh(hdg, n, scale, part)
    with hdg.Context(0) as ctx:
        ctx.set_mesh(m)
        _run(ctx, hdg, 2, hdg.PC_AUTO)  # leaves a hierarchy
        got = _run(ctx, hdg, k, hdg.PC_AUTO)
        ref = _run(ctx, hdg, k, hdg.PC_BLOCK_JACOBI)
        again = _run(ctx, hdg, k, hdg.PC_AUTO)
    print(f"[stretched] {n} k={k} scale={scale} part={part}: {got[0]} iterations, block-Jacobi {ref[0]}", flush=True)
    assert again[0] == got[0] and np.array_equal(again[1], got[1])
    if jacobi:
        assert got[0] == ref[0] and np.array_equal(got[1], ref[1])
    else:
        assert got[0] < 0.8 * ref[0]
