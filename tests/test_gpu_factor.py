"""The deflated Cholesky of the symmetrised Schur matrix and the solve matrices
made from it, at the edges of its 64-wide blocks and 16-wide sub-blocks, and
again on the same plan after the points moved (its workspaces are kept).

Bars: f 1e-10 and s 1e-10 (relative L2) against the oracle; the residual of
S x = b within 1e-11 (a backward-stable solve leaves about cond(M)^(1/2) eps
per block product, cond(M) < 1e6 here: 1e3 x 2.2e-16 x a few tens of products).
"""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


def ring(N, spacing, dx, shift=0.003):
    """N points on a circle `spacing` dx apart (at least 4 dx across), the grid around it."""
    from ilhip import geometry as G
    r = max(N * spacing * dx / (2 * np.pi), 2 * dx)
    n = int(2 * r / dx) + 24
    th = 2 * np.pi * np.arange(N) / N
    s = G.Surface(r * np.cos(th) + shift, r * np.sin(th), np.cos(th), np.sin(th), np.full(N, 2 * np.pi * r / N),
                  np.zeros(N, int))
    return G.GridSpec(n + 1, n + 1, n // 2 + 1, n // 2 + 1, dx), s, th


@pytest.mark.parametrize("N", [1, 2, 16, 17, 64, 65, 66, 128, 129, 130, 193, 321, 450])
def test_factor_block_edges(ctx, N):
    import ilhip
    g, s, th = ring(N, 1.4, 0.02)
    print("factor N", N, "grid", g.NX, flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    b = np.random.default_rng(N).standard_normal(N)
    x = ilhip.SchurFactor(c).solve(b)
    S = ilhip.create_RTLinvR(c)
    assert rel_err(S @ x, b) < 1e-11
    fp, fm = 0.3 + np.cos(th), np.sin(2 * th)
    prob = ilhip.DirichletPoisson(c)
    og = O.grid(g.NX, g.NY, g.I0x, g.I0y, g.dx)
    for shift in (0.003, 0.011):
        t = ring(N, 1.4, 0.02, shift)[1]
        c.update_points(t)
        f, sv = prob.solve(fp, fm, filter_power=0)
        fr, sr = O.dirichlet_solve(og, O.Geometry(t.X, t.Y, t.nx, t.ny, t.ds), fp, fm)
        assert rel_err(f.flat(), fr) < 1e-10
        assert rel_err(sv.flat(), sr) < 1e-10


@pytest.mark.parametrize("N,spacing,ddf", [(33, 1.4, "Roma"), (40, 6.0, "Yang3"), (50, 3.1, "Witchhat"),
                                           (31, 2.0, "M4prime")])
def test_double_layer_assembly(ctx, N, spacing, ddf):
    """E L^-1 D_s for every DDF's window alignment, and for points so far
    apart that a tile's kernel box does not fit in LDS (6 dx)."""
    import ilhip
    g, s, th = ring(N, spacing, 0.02)
    kind = getattr(ilhip, ddf)
    print("double layer N", N, "spacing", spacing, ddf, flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx, ddftype=kind)
    fp = 0.3 + np.cos(th)
    f, sv = ilhip.DirichletPoisson(c).solve(fp, filter_power=0)
    og = O.grid(g.NX, g.NY, g.I0x, g.I0y, g.dx)
    fr, sr = O.dirichlet_solve(og, O.Geometry(s.X, s.Y, s.nx, s.ny, s.ds), fp, ddf_kind=kind)
    assert rel_err(f.flat(), fr) < 1e-10
    assert rel_err(sv.flat(), sr) < 1e-10


@pytest.mark.parametrize("N", [245, 450, 900])
def test_factor_net_charge(ctx, N):
    """The constant mode of S^-1 b for smooth b: sum_p ds_p x_p = q . b with
    S^T q = ds (q refined in extended precision).  The solve's last reflection
    passes its length-N dot's rounding into it, at most N eps |ds x|; the
    factor's own error (thousands of eps, its constant mode being the one that
    f's far field sees) must not show."""
    import ilhip
    g, s, th = ring(N, 1.4, 0.02)
    print("net charge N", N, flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    S = ilhip.create_RTLinvR(c)
    Sl = S.T.astype(np.longdouble)
    inv = np.linalg.inv(S.T)
    q = (inv @ s.ds).astype(np.longdouble)
    for _ in range(4):
        q = q + inv @ (s.ds - Sl @ q).astype(float)
    F = ilhip.SchurFactor(c)
    for b in (0.3 + np.cos(th), np.sin(2 * th) + 0.1 * np.cos(7 * th), np.exp(np.cos(th)), 1 / (1.3 + np.cos(th))):
        x = s.ds * F.solve(b)
        err = abs(float(x.astype(np.longdouble).sum() - q @ b.astype(np.longdouble)))
        print("  error / (eps |x|): %.1f" % (err / (np.finfo(float).eps * np.linalg.norm(x))), flush=True)
        assert err <= N * np.finfo(float).eps * np.linalg.norm(x)


def test_solve_buffers_given_back(ctx):
    """The Dirichlet buffers of the previous geometry wait for a next Dirichlet
    solve for one geometry, and go as soon as the plan takes another solve:
    the factor and the solve matrix are four N x N arrays."""
    import ctypes as C
    import gc

    import ilhip
    N = 1500
    g, s, th = ring(N, 1.4, 0.02)
    moved = ring(N, 1.4, 0.02, 0.011)[1]
    b = 0.3 + np.cos(th)
    mat = 8 * N * N
    print("buffers", flush=True)

    def used():
        gc.collect()
        ctx.synchronize()
        free, total = C.c_size_t(), C.c_size_t()
        assert ilhip.load_library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # from the HIP runtime it links
        return total.value - free.value

    def plan(solve, other):
        c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
        p = ilhip.DirichletPoisson(c)
        p.solve(b, filter_power=0)
        u = [used()]
        c.update_points(moved)
        if solve:
            p.solve(b, filter_power=0)
        u.append(used())
        c.update_points(s)
        if other:
            other(c)
        u.append(used())
        return u

    full, again, moving = plan(True, lambda c: ilhip.DirichletPoisson(c).solve_moving(b))
    assert abs(again - full) < mat   # reused, not allocated beside the old ones
    full, idle, gone = plan(False, None)
    assert abs(idle - full) < mat and gone < full - 3 * mat

    def moving_only():
        c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
        before = used()
        ilhip.DirichletPoisson(c).solve_moving(b)
        return used() - before

    assert moving - full < moving_only() - 3 * mat
