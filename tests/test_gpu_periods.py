"""Source convolutions on the periods their points' extent needs: bodies in the
middle, at an edge, in a corner, thin grids.

Bar: f, s 1e-10 (relative L2) against the oracle.
"""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,cx,cy,r", [(64, 64, 0.5, 0.5, 8), (65, 33, 0.5, 0.5, 8), (100, 140, 0.0, 0.5, 12),
                                         (129, 70, 1.0, 1.0, 9), (200, 97, 0.0, 0.0, 20), (260, 60, 0.3, 0.5, 14),
                                         (150, 600, 0.5, 0.9, 30),
                                         (140, 64, 0.9172, 0.5, 20)])   # last: the primal and dual periods differ
def test_source_periods(ctx, n, m, cx, cy, r):
    """A circle of r cells, its centre at the fraction (cx, cy) between the
    positions that keep it 6 cells inside the grid."""
    import ilhip
    from ilhip import geometry as G
    dx = 0.02
    g = G.GridSpec(n + 1, m + 1, n // 2 + 1, m // 2 + 1, dx)
    lo = r + 6
    x = g.x_primal()[0] + (lo + cx * (n - 1 - 2 * lo)) * dx
    y = g.y_primal()[0] + (lo + cy * (m - 1 - 2 * lo)) * dx
    s = G.circle(r * dx, 1.4 * dx, x, y)
    print("periods", n, m, "centre", x / dx, y / dx, "N", s.N, flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    og, geo = O.grid(g.NX, g.NY, g.I0x, g.I0y, dx), O.Geometry(s.X, s.Y, s.nx, s.ny, s.ds)
    th = s.theta(x, y)
    fp, fm = np.cos(th) + 0.2, np.sin(2 * th)
    f, sv = ilhip.DirichletPoisson(c).solve(fp, fm, filter_power=0)
    fr, sr = O.dirichlet_solve(og, geo, fp, fm)
    assert rel_err(f.flat(), fr) < 1e-10
    assert rel_err(sv.flat(), sr) < 1e-10
    f, df, st, ds = ilhip.NeumannPoisson(c).solve(fp, fm)
    for a, b in zip((f, df, st, ds), O.neumann_solve(og, geo, fp, fm)):
        assert rel_err(a.flat(), b) < 1e-10


def test_batch_of_small_and_centred(ctx):
    """A body in the middle of 48 cells needs a period of 64, below the fused
    batch's 128, and one in the middle of 140 x 300 needs half the grid's: the
    batch is fused all the same and equals the single solves bit for bit."""
    import ilhip
    from ilhip import geometry as G
    dx = 0.02
    caches, fbs = [], []
    for n, m, r in ((48, 48, 6), (140, 300, 12), (60, 52, 7)):
        g = G.GridSpec(n + 1, m + 1, n // 2 + 1, m // 2 + 1, dx)
        s = G.circle(r * dx, 1.4 * dx, 0.3 * dx, -0.2 * dx)
        caches.append(ilhip.SurfaceScalarCache(s, g, ctx=ctx))
        fbs.append(np.cos(s.theta(0, 0)) + 0.2)
    print("fused batch of small grids", flush=True)
    out = ilhip.dirichlet_solve_batched(caches, fbs)
    fp = [ilhip.DeviceArray.from_host(ctx, b) for b in fbs]
    fd = [ilhip.DeviceArray(ctx, int(np.prod(c.g.primal_shape()))) for c in caches]
    sd = [ilhip.DeviceArray(ctx, len(b)) for b in fbs]
    batch = ilhip.DirichletBatch(caches, fp, fd, sd)
    print("tuning", batch.tuning(), flush=True)   # an error for a batch of single launches
    batch.launch()
    ctx.synchronize()
    for k, c in enumerate(caches):
        f, s = ilhip.DirichletPoisson(c).solve(fbs[k], filter_power=0)
        for a, b in ((out[k][0].flat(), f.flat()), (out[k][1].flat(), s.flat()), (fd[k].download(), f.flat()),
                     (sd[k].download(), s.flat())):
            assert np.array_equal(a, b)
