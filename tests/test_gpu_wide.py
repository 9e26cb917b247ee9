"""A flat grid wider than the marching kernels have blocks (2048 windows of 62
columns, 126,976 points): their blocks take a second window.  The trace is
checked on the host against the exported matrix, as for the reduced system's
other shapes; with two square cells across, cond(K) is of order 10 and CG's 1e-12
of the load is what is left, so the bound of 1e-11 is wide."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,k,precision", [(126900, 1, 0), (130000, 1, 0), (127100, 2, 1)])
def test_second_window(hdg, nx, k, precision):
    print(f"[wide] {nx}x2 k={k} precision={precision}", flush=True)
    m = hdg.rectangle_mesh((nx, 2))
    m = hdg.PolygonalMesh(m.nodes * [0.5 * nx, 1.0], m.cells, m.faces, m.facesets, m.nodesets)
    with hdg.Context(0) as ctx:
        ctx.set_mesh(m)
        ctx.setup(k, quad_degree=k + 1, rtol=1e-12, precision=precision)
        ctx.set_source()
        d = m.boundary_dofs(k + 1)
        v = np.cos(np.arange(len(d)))
        ctx.set_dirichlet(d, v)
        info = ctx.run()
        x = ctx.trace()
        K, b = ctx.get_system_scipy()
    free = np.ones(len(x), dtype=bool)
    free[d - 1] = False
    assert np.array_equal(x[~free], v)
    lift = np.where(free, 0.0, x)
    res = np.linalg.norm((b - K @ x)[free]) / np.linalg.norm((b - K @ lift)[free])
    print(f"    {info.iters} iterations, residual {res:.1e}", flush=True)
    assert res < 1e-11 and info.true_relres < 1e-11
