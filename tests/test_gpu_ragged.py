"""Vertex levels with odd sides (a last coarse column or row one fine cell
wide, on one level or on several), Dirichlet data on the whole boundary or on
one side of it: CG's iteration count against the same method written with
scipy from the exported matrix (diagonals eliminated, Galerkin products of
the same interpolation, the same sweeps).  A wrong coarse stencil changes
the count; rounding does not.  The smoothing weights may differ: both come
from four Lanczos steps behind a random load, which put the largest eigenvalue
within a few per cent, worth an iteration either way; the bound is two."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

pytestmark = pytest.mark.gpu

RTOL = 1e-10


def _interp(n):
    """coarse to fine, one dimension: n cells from (n + 1) // 2."""
    x = np.arange(n + 1)
    own = (x % 2 == 0) | (x == n)
    lo = np.where(x == n, (n + 1) // 2, x // 2)
    hi = np.where(own, lo, lo + 1)
    r = np.concatenate([x, x])
    return sp.csr_matrix((np.full(2 * n + 2, 0.5), (r, np.concatenate([lo, hi]))), shape=(n + 1, (n + 1) // 2 + 1))


def _reference(m, nx, ny, nt, K, b, d, factor):
    n = len(b)
    free = np.ones(n, dtype=bool)
    free[d - 1] = False
    f = m.faces
    diag = (f[:, 3] > 0) & ((f[:, 2] - 1) // 2 == (f[:, 3] - 1) // 2)
    isd = np.repeat(diag, nt)
    S, b = -K.tocsr(), -b
    o, q = np.nonzero(free & ~isd)[0], np.nonzero(free & isd)[0]
    lu = spl.splu(S[q][:, q].tocsc())
    Soq, Sqo = S[o][:, q], S[q][:, o].tocsc()
    inv = sp.csc_matrix(lu.solve(np.eye(len(q)))) if len(q) < 600 else None
    if inv is None:  # nt x nt blocks
        blk = [np.linalg.inv(S[q[i:i + nt]][:, q[i:i + nt]].toarray()) for i in range(0, len(q), nt)]
        inv = sp.block_diag(blk, format="csc")
    T = (S[o][:, o] - Soq @ inv @ Sqo).tocsr()
    r = b[o] - Soq @ (inv @ b[q])
    # block-Jacobi over the faces
    face = o // nt
    start = np.concatenate([[0], np.nonzero(np.diff(face))[0] + 1, [len(o)]])
    J = sp.block_diag([np.linalg.inv(T[i:j][:, i:j].toarray()) for i, j in zip(start[:-1], start[1:])], format="csr")
    # Lanczos by block-Jacobi CG
    rng = np.random.default_rng(1)
    x = rng.uniform(-1, 1, len(o))
    z = J @ x
    p, rz, al, be = z, x @ z, [], []
    for _ in range(4):
        Tp = T @ p
        al.append(rz / (p @ Tp))
        x = x - al[-1] * Tp
        z = J @ x
        rz, old = x @ z, rz
        be.append(rz / old)
        p = z + be[-1] * p
    M = np.diag([1 / al[i] + (be[i - 1] / al[i - 1] if i else 0) for i in range(4)])
    for i in range(3):
        M[i, i + 1] = M[i + 1, i] = np.sqrt(be[i]) / al[i]
    om = factor / np.linalg.eigvalsh(M)[-1]
    # vertex levels
    ends = f[face, :2] - 1
    lo, hi, mode = ends.min(axis=1), ends.max(axis=1), o % nt
    nv = (nx + 1) * (ny + 1)
    w = np.where(mode == 0, 0.5, np.where(mode == 1, -1 / (2 * np.sqrt(3)), 0.0))
    P = sp.csr_matrix((np.concatenate([w, np.abs(w)]), (np.tile(np.arange(len(o)), 2), np.concatenate([lo, hi]))),
                      shape=(len(o), nv))
    fixed = np.zeros(nv, dtype=bool)
    pf = (d[(d - 1) % nt == 0] - 1) // nt
    fixed[(f[pf[~diag[pf]], :2] - 1).ravel()] = True
    P = (P @ sp.diags((~fixed).astype(float))).tocsr()
    As, Ps, cx, cy = [], [P], nx, ny
    A = (P.T @ T @ P).tocsr()
    while True:
        A = A + sp.diags(fixed.astype(float))
        As.append(A.tocsr())
        if (cx + 1) * (cy + 1) <= 96:
            break
        gx, gy = np.minimum(2 * np.arange((cx + 1) // 2 + 1), cx), np.minimum(2 * np.arange((cy + 1) // 2 + 1), cy)
        Q = sp.kron(_interp(cy), _interp(cx))
        cf = fixed.reshape(cy + 1, cx + 1)[np.ix_(gy, gx)].ravel()
        Q = (sp.diags((~fixed).astype(float)) @ Q @ sp.diags((~cf).astype(float))).tocsr()
        free_l = sp.diags((~fixed).astype(float))
        A = (Q.T @ (free_l @ A @ free_l) @ Q).tocsr()
        Ps.append(Q)
        fixed, cx, cy = cf, (cx + 1) // 2, (cy + 1) // 2
    bottom = spl.splu(As[-1].tocsc())

    def vc(level, g):
        if level == len(As) - 1:
            return bottom.solve(g)
        D = 0.7 / As[level].diagonal()
        e = D * g
        e = e + Ps[level + 1] @ vc(level + 1, Ps[level + 1].T @ (g - As[level] @ e))
        return e + D * (g - As[level] @ e)

    def cycle(g):
        e = om * (J @ g)
        e = e + P @ vc(0, P.T @ (g - T @ e))
        return e + om * (J @ (g - T @ e))

    stop = RTOL * np.linalg.norm(b[free])
    z = cycle(r)
    p, rz = z, r @ z
    for it in range(1, 200):
        Tp = T @ p
        a = rz / (p @ Tp)
        r = r - a * Tp
        if np.linalg.norm(r) <= stop:
            return it
        z = cycle(r)
        rz, old = r @ z, rz
        p = z + rz / old * p
    return 200


@pytest.mark.parametrize("one_side", [False, True])
@pytest.mark.parametrize("nx,ny,k", [(17, 31, 1), (33, 9, 2), (65, 47, 3), (65, 65, 1), (40, 27, 4), (95, 33, 2)])
def test_odd_sides(hdg, nx, ny, k, one_side):
    print(f"[ragged] {nx}x{ny} k={k} one_side={one_side}", flush=True)
    m = hdg.rectangle_mesh((nx, ny))
    nt = k + 1
    d = m.boundary_dofs(nt)
    if one_side:
        low = np.nonzero((m.nodes[m.faces[:, :2] - 1][:, :, 1] == 0.0).all(axis=1))[0]
        d = d[np.isin((d - 1) // nt, low)]
    with hdg.Context(0) as ctx:
        ctx.set_mesh(m)
        ctx.setup(k, quad_degree={1: 2, 2: 3, 3: 6, 4: 6}[k], rtol=RTOL)
        ctx.set_source()
        ctx.set_dirichlet(d, np.zeros(len(d)))
        its = ctx.run().iters
        K, b = ctx.get_system_scipy()
    ref = _reference(m, nx, ny, nt, K, b, d, 1.27 if k % 2 else 1.42)
    assert abs(its - ref) <= 2, (its, ref)
