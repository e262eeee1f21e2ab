"""The Stokes solve where its launches differ: bodies at the edge of the allowed
margin, thin grids, odd and even point counts, source periods below the grid's
own (which the potential always takes), other DDFs.

Bars as the vector cache's Stokes tests: relative L2 1e-10 for the velocity and
for the streamfunction up to a constant, 1e-9 for the traction.
"""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,r,px,py,npts,ddf", [
    (64, 64, 10, 0.5, 0.5, 41, "yang3"), (64, 64, 10, 0.0, 1.0, 42, "yang3"), (45, 120, 9, 1.0, 0.3, 37, "yang3"),
    (141, 60, 14, 0.93, 0.0, 57, "roma"), (90, 66, 12, 0.0, 0.5, 50, "m4prime"), (70, 70, 9, 1.0, 1.0, 35, "yang3")])
def test_stokes_sizes(ctx, nx, ny, r, px, py, npts, ddf):
    """npts points on a circle of r cells, its centre at the fraction (px, py)
    between the positions that keep the supports just inside the margin."""
    import ilhip
    from ilhip import geometry as G
    dx = 0.05
    gs = G.GridSpec(nx, ny, nx // 2, ny // 2, dx)
    lo = r + 8
    x0, y0 = gs.x_primal()[0], gs.y_primal()[0]
    cx, cy = x0 + (lo + px * (nx - 2 - 2 * lo)) * dx, y0 + (lo + py * (ny - 2 - 2 * lo)) * dx
    s = G.circle(r * dx, 2 * np.pi * r * dx / npts, cx, cy)
    print("stokes", nx, ny, "N", s.N, ddf, flush=True)
    kind = {"yang3": O.YANG3, "roma": O.ROMA, "m4prime": O.M4PRIME}[ddf]
    c = ilhip.SurfaceVectorCache(s, gs, ctx=ctx, ddftype=kind)
    og, geo = O.grid(gs.NX, gs.NY, gs.I0x, gs.I0y, dx), O.Geometry(s.X, s.Y, s.nx, s.ny, s.ds)
    th = s.theta(cx, cy)
    vp = np.concatenate([np.cos(th) + 0.3, np.sin(2 * th)])
    vm = np.concatenate([0.2 * np.sin(th), np.cos(3 * th)])
    prob = ilhip.StokesFlow(c)
    for minus in (None, vm):
        rv, rs, rsig = O.stokes_solve(og, geo, vp, minus, ddf_kind=kind)
        Cf = O.surface_filter_vector(og, geo, ddf_kind=kind)
        for power in (0, 1, 2, 3):
            v, st, sig = prob.solve(vp, minus, filter_power=power)
            assert rel_err(v.flat(), rv) < 1e-10
            d = st.flat() - rs
            assert rel_err(st.flat() - d.mean(), rs) < 1e-10
            assert rel_err(sig.flat(), np.linalg.matrix_power(Cf, power) @ rsig) < 1e-9


def test_stokes_new_geometry(ctx):
    """A plan whose points moved (its source buffers are kept), to more and to
    fewer grid rows, equals a fresh plan bit for bit."""
    import ilhip
    from ilhip import geometry as G
    dx = 0.05
    gs = G.GridSpec(90, 80, 45, 40, dx)
    th = 2 * np.pi * np.arange(44) / 44

    def body(a, b):
        w = np.hypot(a * np.sin(th), b * np.cos(th))
        return G.Surface(a * dx * np.cos(th), b * dx * np.sin(th), b * np.cos(th) / w, a * np.sin(th) / w,
                         w * dx * 2 * np.pi / 44, np.zeros(44, int))

    vp = np.concatenate([np.cos(th) + 0.3, np.sin(2 * th)])
    c = ilhip.SurfaceVectorCache(body(10, 8), gs, ctx=ctx)
    prob = ilhip.StokesFlow(c)
    prob.solve(vp, filter_power=2)
    for a, b in ((6, 15), (14, 5)):
        print("stokes moved to", a, b, flush=True)
        c.update_points(body(a, b))
        got = prob.solve(vp, filter_power=2)
        want = ilhip.StokesFlow(ilhip.SurfaceVectorCache(body(a, b), gs, ctx=ctx)).solve(vp, filter_power=2)
        for x, y in zip(got, want):
            assert np.array_equal(x.flat(), y.flat())
