"""A source that is refused leaves the one before it in place: values that the
call lacks (no pointer) or has no room for (budget).  The next run solves with
the old source, bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(hdg, k, precond, budget=0):
    ctx = hdg.Context(0, hbm_budget=budget)
    ctx.set_rectangle_mesh(13, 9, jitter=0.2, seed=k)
    ctx.setup(k, quad_degree=2 if k == 1 else 3, precond=precond)
    ctx.set_dirichlet_boundary(0.0)
    return ctx


@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("precond", [0, 1])
def test_refused_source(hdg, k, precond):
    L = hdg._lib
    with _context(hdg, k, precond) as ctx:
        f = np.random.default_rng(k).standard_normal((2 * 13 * 9, ctx.sizes.nqp))
        ctx.set_source(kind=3, f_qp=f)
        ctx.run()
        u = ctx.trace()
        s = L.Source()
        s.kind = 3  # and no values
        with pytest.raises(hdg.HDGError, match="f_qp"):
            L.check(L.lib().hdg_set_source(ctx._h, C.byref(s)), ctx._h)
        ctx.run()
        assert np.array_equal(ctx.trace(), u)
        ctx.set_source()
        ctx.run()
        v = ctx.trace()
        ctx.set_source(kind=3, f_qp=f)
        ctx.set_source(kind=3, f_qp=2.0 * f)  # over the old values
        ctx.run()
        assert np.array_equal(ctx.trace(), 2.0 * u) and not np.array_equal(v, u)


def test_source_without_room(hdg):
    with _context(hdg, 2, 1) as ctx:
        ctx.set_source()
        ctx.run()
        u, used = ctx.trace(), ctx.memory_used()
    with _context(hdg, 2, 1, budget=used) as ctx:
        ctx.set_source()
        ctx.run()
        with pytest.raises(hdg.HDGError, match="budget"):
            ctx.set_source(kind=3, f_qp=np.ones((2 * 13 * 9, ctx.sizes.nqp)))
        assert np.array_equal(ctx.trace(), u)
        ctx.run()
        assert np.array_equal(ctx.trace(), u)
