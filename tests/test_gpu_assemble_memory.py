"""hdg_assemble_condense on a rectangle mesh makes what the solve reads, the
condensed cells, and leaves the assembled matrix to the exports: no memory for
it before one is asked for, and under a budget that holds the solve alone,
assembling and solving in turn gives hdg_run's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QD = {1: 2, 2: 3, 3: 6, 4: 6}


def _context(hdg, k, budget=0):
    ctx = hdg.Context(0, hbm_budget=budget)
    ctx.set_rectangle_mesh(31, 28, jitter=0.2, seed=k)
    ctx.setup(k, quad_degree=QD[k])
    ctx.set_source()
    ctx.set_dirichlet_boundary(0.5)
    return ctx


@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_no_matrix_for_the_solve(hdg, k):
    with _context(hdg, k) as ctx:
        ctx.run()
        u, used = ctx.trace(), ctx.memory_used()
        K, b = ctx.get_system_scipy()
        assert ctx.memory_used() > used
    with _context(hdg, k, budget=used) as ctx:
        for _ in range(3):
            ctx.assemble_condense()
            assert ctx.memory_used() == used
            v, _ = ctx.solve()
            assert np.array_equal(u, v) and ctx.memory_used() == used
    with _context(hdg, k) as ctx:
        ctx.assemble_condense()
        K1, b1 = ctx.get_system_scipy()
        v, _ = ctx.solve()
        assert np.array_equal(K.data, K1.data) and np.array_equal(b, b1) and np.array_equal(u, v)
