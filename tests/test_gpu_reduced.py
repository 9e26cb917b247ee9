"""The reduced trace system of rectangle meshes (the diagonal faces eliminated
exactly) where its kernels' partitions can go wrong: fewer columns than the
62 a wavefront owns, just as many, one more; one row, fewer rows than a block
walks, many; every order; tau = 1 (the product acts on differences) and not;
boundary data; and prescribed dofs on diagonal and axis faces inside the
domain.  The trace solution is checked on the host against the assembled
matrix and rhs exported from the device (poisson2D_HDG.jl:176-195), in
which nothing is eliminated: relative residual on the free rows, and the
prescribed rows exactly.  CG stops at 1e-13 of the load; the FP64 floor of
that residual, eps ||K|| ||uhat|| / ||b|| ~ eps cond(K) ~ 2e-16 * 8 n^2, is
below 5e-11 for n <= 160 cells along the shorter side."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _diagonal_faces(m):
    """0-based faces shared by the two triangles of a grid cell."""
    f = m.faces
    return np.nonzero((f[:, 3] > 0) & ((f[:, 2] - 1) // 2 == (f[:, 3] - 1) // 2))[0]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,k,tau,inside", [
    (1, 1, 1, 1.0, False), (2, 1, 4, 1.0, False), (1, 5, 2, 3.0, False), (61, 3, 3, 1.0, False),
    (62, 4, 1, 1.0, False), (63, 5, 2, 0.5, False), (124, 9, 4, 1.0, False), (125, 1, 3, 1.0, False),
    (7, 66, 4, 2.0, False), (160, 130, 1, 1.0, False), (97, 81, 3, 1.0, False),
    (6, 5, 1, 1.0, True), (30, 17, 2, 1.0, True), (64, 23, 3, 2.0, True), (12, 40, 4, 1.0, True),
    (1, 5, 2, 0.3, False), (7, 66, 4, 0.5, False), (64, 23, 3, 0.5, True)])
def test_reduced_system_solution(hdg, nx, ny, k, tau, inside, precision):
    print(f"[reduced] {nx}x{ny} k={k} tau={tau} inside={inside} precision={precision}", flush=True)
    rng = np.random.default_rng(nx * 1000 + ny)
    m = hdg.rectangle_mesh((nx, ny), jitter=0.2, seed=nx + ny)
    nt = k + 1
    dofs = list(m.boundary_dofs(nt))
    if inside:
        d = rng.choice(_diagonal_faces(m), size=3, replace=False)
        inner = np.setdiff1d(np.nonzero(m.faces[:, 3] > 0)[0], _diagonal_faces(m))
        a = rng.choice(inner, size=2, replace=False)
        # one whole diagonal face, single modes of the others
        dofs += [int(d[0]) * nt + t + 1 for t in range(nt)]
        dofs += [int(d[1]) * nt + 1, int(d[2]) * nt + nt, int(a[0]) * nt + 1, int(a[1]) * nt + 2]
    dofs = np.array(sorted(dofs))
    vals = rng.uniform(-1.0, 1.0, len(dofs))
    with hdg.Context(0) as ctx:
        ctx.set_mesh(m)
        ctx.setup(k, quad_degree=QD[k], tau=tau, rtol=1e-13, precision=precision)
        ctx.set_source()
        ctx.set_dirichlet(dofs, vals)
        if tau > 1.0:
            # the reference's H carries no tau (poisson2D_HDG.jl:149): -K is
            # indefinite for tau > 1 on these meshes, and CG reports it
            with pytest.raises(hdg.HDGError, match="broke down"):
                ctx.run()
            return
        info = ctx.run()
        u = ctx.trace()
        colptr, rowval, nzval, rhs = ctx.get_system()
        # solving again on the assembled operators gives the same bits
        ctx.assemble_condense()
        u2, _ = ctx.solve()
    assert np.array_equal(u, u2)
    n = len(rhs)
    K = sp.csc_matrix((nzval, rowval - 1, colptr - 1), shape=(n, n))
    free = np.ones(n, dtype=bool)
    free[dofs - 1] = False
    assert np.array_equal(u[~free], vals)
    uD = np.where(free, 0.0, u)
    b = (rhs - K @ uD)[free]
    res = np.linalg.norm((K @ u - rhs)[free]) / np.linalg.norm(b)
    print(f"    {info.iters} iterations, host residual {res:.2e}, device {info.true_relres:.2e}", flush=True)
    assert res < 5e-11 and info.true_relres < 5e-11
