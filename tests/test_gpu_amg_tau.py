"""Stabilisations on a mesh without rectangle structure: which are solved and
which are refused, by either preconditioner.  The reference's H carries no tau
(poisson2D_HDG.jl:149), so above tau = 1 the cells' blocks lose their
semidefiniteness and, from about 1.2 on this mesh, -K its definiteness, which CG
reports as a breakdown; nothing else may stop a solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _mesh(hdg):
    m = hdg.rectangle_mesh((21, 23), jitter=0.15, seed=21)
    p = np.random.default_rng(21).permutation(len(m.cells))
    faces = m.faces.copy()
    faces[:, 2:] = np.concatenate([[0], np.argsort(p) + 1])[faces[:, 2:]]
    r, t = 1.0 - 0.6 * m.nodes[:, 0], np.pi * m.nodes[:, 1]
    return hdg.PolygonalMesh(np.stack([r * np.cos(t), -r * np.sin(t)], axis=1), m.cells[p], faces, m.facesets, m.nodesets)


@pytest.mark.parametrize("tau,solved", [(0.001, True), (0.3, True), (1.0, True), (1.03, True), (1.3, False), (3.0, False),
                                        (30.0, False)])
@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_outcome(hdg, k, tau, solved):
    m = _mesh(hdg)
    its = []
    for precond in (hdg.PC_BLOCK_JACOBI, hdg.PC_AUTO):
        with hdg.Context(0) as ctx:
            ctx.set_mesh(m)
            ctx.setup(k, quad_degree=QD[k], tau=tau, precond=precond)
            ctx.set_source()
            ctx.set_dirichlet_boundary(0.0)
            if not solved:
                with pytest.raises(hdg.HDGError, match="broke down"):
                    ctx.run()
                continue
            its.append(ctx.run().iters)
    if solved:
        print(f"[tau] k={k} tau={tau}: {its[1]} iterations, block-Jacobi {its[0]}")
        assert its[1] <= 80 and its[1] < its[0] // 2
