"""Heat conduction on the tiled one-kernel filter and the packed stage inverses,
at the edges of the 64 x 64 tiles and of the filter widths (8 to 16 taps a
side, then the two-pass form), with a body 5 cells from the grid's edge, new
boundary values between calls, and without bodies.

Bar: 1e-11 (relative L2) against the oracle: stage matrices of condition < 50
at these points and Fourier numbers (140 at 1.6), three solves and six filters a step, at
most 5 steps: a few hundred roundings of 1e-16.
"""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,fo,N", [(63, 64, 0.02, 40), (64, 65, 0.1, 60), (129, 70, 0.25, 70), (100, 140, 0.45, 90),
                                      (193, 128, 0.62, 120), (90, 91, 0.9, 64), (70, 129, 0.25, 0),
                                      # the shorter filter alone has at most 16 taps a side
                                      (97, 130, 1.2, 80), (130, 66, 1.6, 70), (70, 129, 1.3, 0)])
def test_heat_tiles(ctx, n, m, fo, N):
    import ilhip
    from ilhip import geometry as G
    dx = 0.02
    g = G.GridSpec(n + 1, m + 1, n // 2 + 1, m // 2 + 1, dx)
    r = N * 1.4 * dx / (2 * np.pi)
    th = 2 * np.pi * np.arange(N) / max(N, 1)
    # leftmost point 5.3 cells from the grid's left edge, centre a little off the cells
    cx, cy = g.x_primal()[0] + 5.3 * dx + r, 0.4 * dx
    s = G.Surface(cx + r * np.cos(th), cy + r * np.sin(th), np.cos(th), np.sin(th), np.full(N, 1.4 * dx),
                  np.zeros(N, int))
    rng = np.random.default_rng(n)
    T0 = rng.standard_normal((n, m))
    print("heat tiles", n, m, "Fo", fo, "N", N, flush=True)
    og = O.grid(g.NX, g.NY, g.I0x, g.I0y, dx)
    geo = O.Geometry(s.X, s.Y, s.nx, s.ny, s.ds)
    tp, tm = 1.0 + 0.3 * np.cos(th), 0.2 * np.sin(3 * th)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    heat = ilhip.DirichletHeatConduction(c, 1.0, fo * dx * dx, tp, tm)
    T = ilhip.Nodes(ilhip.Primal, g, T0.copy())
    ref = T0.ravel(order="F").copy()
    for k, (a, b, steps) in enumerate(((tp, tm, 2), (tm, None, 1), (tp - tm, tp, 2))):
        if k:
            heat.set_boundary(a, b)
        heat.advance(T, steps)
        ref = O.heat_advance(og, geo, 1.0, fo * dx * dx, steps, ref, a, b if b is not None else np.zeros(N))
        assert rel_err(T.flat(), ref) < 1e-11
        if N:
            Eb = ilhip.ScalarData(N)
            ilhip.interpolate(Eb, T, c)
            assert np.abs(Eb.flat() - 0.5 * (a + (0 if b is None else b))).max() < 1e-12
    heat.close()


@pytest.mark.parametrize("N", [30, 47, 64, 90])
def test_heat_first_point_twice(ctx, N):
    """Two points at one place: the stage matrices are singular, and the last
    pivots of their factorisation (the first point's among them) are rounding
    of either sign, which must not pass for a positive one."""
    import ilhip
    from ilhip import geometry as G
    dx = 0.02
    g = G.GridSpec(131, 111, 66, 56, dx)
    r = N * 1.4 * dx / (2 * np.pi)
    th = np.concatenate([[0.0], 2 * np.pi * np.arange(N) / N])
    ds = np.full(N + 1, 1.4 * dx)
    ds[:2] *= 0.5
    for shift in (0.0, 0.003, 0.0071):
        s = G.Surface(r * np.cos(th) + shift, r * np.sin(th), np.cos(th), np.sin(th), ds, np.zeros(N + 1, int))
        c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
        for fo in (0.1, 0.5, 1.0):
            print("heat, one point twice", N, shift, fo, flush=True)
            with pytest.raises(ilhip.SingularError):
                ilhip.DirichletHeatConduction(c, 1.0, fo * dx * dx, np.cos(th))
