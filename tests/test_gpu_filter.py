"""The surface filter's three routes -- one work-group, one launch a power, the
grid (rows of more than 64 entries) -- on host and device memory, in place and
not, against C built by create_surface_filter.  Bar 1e-12 (max-abs relative),
the filter's bar elsewhere.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import max_rel

pytestmark = pytest.mark.gpu


# points, radius in cells: one point, two far apart, around a wave and a
# work-group, the longest one work-group takes and one more, a dense sampling
@pytest.mark.parametrize("npts,r", [(1, 8.0), (2, 9.0), (63, 14.0), (64, 14.5), (1025, 240.0), (2048, 480.0),
                                    (2049, 480.0), (4096, 950.0), (4097, 950.0), (300, 6.0)])
def test_filter_routes(ctx, npts, r):
    import ilhip
    import ilhip._lib as L
    from ilhip import geometry as G
    n = int(2 * r) + 16
    dx = 1.0 / n
    g = G.GridSpec(n, n, n // 2, n // 2, dx)
    th = 2 * np.pi * (np.arange(npts) + 0.3) / npts
    ds = np.full(npts, 2 * np.pi * r * dx / npts)
    s = G.Surface(r * dx * np.cos(th), r * dx * np.sin(th), np.cos(th), np.sin(th), ds, np.zeros(npts, int))
    print("filter", npts, "points, radius", r, flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    Cm = ilhip.create_surface_filter(c)
    longest = int((Cm != 0).sum(axis=1).max())
    assert (longest > 64) == (npts == 300)
    x = np.random.default_rng(npts).standard_normal(npts)
    ref = x
    dev, out = ilhip.DeviceArray.from_host(ctx, x), ilhip.DeviceArray(ctx, npts)
    for k in range(4):
        assert max_rel(ilhip.filter_surface(ilhip.ScalarData(npts, x), c, k).flat(), ref) < 1e-12
        L.call("ilh_surface_filter_apply", c.h, k, dev.ptr, out.ptr, L.MEM_DEVICE)
        assert max_rel(out.download(), ref) < 1e-12
        ip = ilhip.DeviceArray.from_host(ctx, x)
        L.call("ilh_surface_filter_apply", c.h, k, ip.ptr, ip.ptr, L.MEM_DEVICE)
        assert max_rel(ip.download(), ref) < 1e-12
        ref = Cm @ ref
    # a new geometry takes new rows
    m = G.Surface(s.X + 0.3 * dx, s.Y - 0.4 * dx, s.nx, s.ny, s.ds, s.body)
    c.update_points(m)
    got = ilhip.filter_surface(ilhip.ScalarData(npts, x), c, 2).flat()
    Cm = ilhip.create_surface_filter(c)
    assert max_rel(got, Cm @ (Cm @ x)) < 1e-12


def test_filter_rows_too_long_in_one_place(ctx):
    """An ordinary mean spacing with one crowded arc (300 of 600 points on 20
    cells): found on the device, and the grid takes over."""
    import ilhip
    from ilhip import geometry as G
    n, dx, r = 140, 0.01, 60.0
    arc = 20.0 / r
    edges = np.concatenate([np.linspace(0, arc, 301), np.linspace(arc, 2 * np.pi, 301)[1:]])
    th, w = 0.5 * (edges[1:] + edges[:-1]), np.diff(edges)
    g = G.GridSpec(n, n, n // 2, n // 2, dx)
    s = G.Surface(r * dx * np.cos(th), r * dx * np.sin(th), np.cos(th), np.sin(th), r * dx * w, np.zeros(600, int))
    print("filter, one crowded arc", flush=True)
    c = ilhip.SurfaceScalarCache(s, g, ctx=ctx)
    Cm = ilhip.create_surface_filter(c)
    assert int((Cm != 0).sum(axis=1).max()) > 64
    x = ref = np.random.default_rng(7).standard_normal(600)
    for k in range(3):
        assert max_rel(ilhip.filter_surface(ilhip.ScalarData(600, x), c, k).flat(), ref) < 1e-12
        ref = Cm @ ref
