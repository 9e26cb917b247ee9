"""The pinned memory of exports is the process's, lent to one export at a time:
more contexts than it keeps pieces for export side by side from threads of their
own, results below, at and beyond one piece, and every array arrives whole; then
again on new contexts after all of these have gone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(3, 2, 1), (40, 33, 2), (64, 61, 3), (150, 171, 1), (90, 83, 4)]


def test_side_by_side(hdg):
    for _ in range(2):
        bad = []

        def work(i):
            try:
                nx, ny, k = SIZES[i % len(SIZES)]
                with hdg.Context(0) as ctx:
                    ctx.set_rectangle_mesh(nx, ny, jitter=0.2, seed=i)
                    ctx.setup(k, quad_degree={1: 2, 2: 3, 3: 6, 4: 6}[k])
                    ctx.set_source()
                    ctx.set_dirichlet_boundary(0.0)
                    ctx.assemble_condense()
                    s = ctx.sizes
                    first = None
                    for r in range(6):
                        x = np.random.default_rng(100 * i + r).standard_normal(s.n_dofs)
                        ctx.set_trace(x)
                        if not np.array_equal(ctx.trace(), x):
                            bad.append((i, r, "trace"))
                        K, b = ctx.get_system_scipy()
                        Ke, be = ctx.get_local_ops()
                        got = (K.indptr, K.indices, K.data, b, Ke, be)
                        first = first or got
                        if not all(np.array_equal(p, q) for p, q in zip(first, got)):
                            bad.append((i, r, "system"))
            except Exception as e:  # noqa: BLE001
                bad.append((i, repr(e)))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(12)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad, bad
