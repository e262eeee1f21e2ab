"""The moving solve's Arnoldi step, which one work-group does alone for the
first steps (16 up to 2048 points, 8 up to 4096, none above) and slices of 64
points after that: trajectories of very different sizes in one batch, on both
sides of both limits, so that steps 0 to 15 run both kernels at once, equal
their single solves bit for bit, and f agrees with a fresh direct solve to the
FP64 bar (relative L2 1e-10).
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _bodies():
    from ilhip import geometry as G
    out = []
    for n, r, spacing in ((80, 10.0, 1.4), (400, 163.0, 1.0), (400, 163.6, 1.0), (760, 326.1, 1.0),
                          (760, 326.3, 1.0), (1420, 652.0, 1.0), (1420, 652.2, 1.0)):
        dx = 2.0 / n
        g = G.GridSpec(n + 1, n + 1, n // 2, n // 2, dx)
        out.append((g, G.circle(r * dx, spacing * dx, 0.3 * dx, -0.2 * dx)))
    return out


def test_batch_of_mixed_sizes(ctx):
    import ilhip
    from ilhip import geometry as G
    bodies = _bodies()
    print("points", [s.N for _, s in bodies], flush=True)
    assert [s.N for _, s in bodies] == [44, 1024, 1027, 2048, 2050, 4096, 4097]
    fbs = [np.cos(s.theta(0, 0)) + 0.3 * np.sin(5 * s.theta(0, 0)) for _, s in bodies]
    cb = [ilhip.SurfaceScalarCache(s, g, ctx=ctx) for g, s in bodies]
    cs = [ilhip.SurfaceScalarCache(s, g, ctx=ctx) for g, s in bodies]
    fp = [ilhip.DeviceArray.from_host(ctx, x) for x in fbs]
    fd = [ilhip.DeviceArray(ctx, int(np.prod(g.primal_shape()))) for g, _ in bodies]
    sd = [ilhip.DeviceArray(ctx, s.N) for _, s in bodies]
    ilhip.dirichlet_solve_moving_batched(cb, fp, fd, sd, tol=1e-12, max_iter=200)
    for c, x in zip(cs, fbs):
        ilhip.DirichletPoisson(c).solve_moving(x, tol=1e-12, max_iter=200)
    moved = [G.Surface(s.X + 0.35 * g.dx, s.Y - 0.2 * g.dx, s.nx, s.ny, s.ds, s.body) for g, s in bodies]
    for k, m in enumerate(moved):
        cb[k].update_points(m)
        cs[k].update_points(m)
    its = ilhip.dirichlet_solve_moving_batched(cb, fp, fd, sd, tol=1e-12, max_iter=200)
    ctx.synchronize()
    # steps 8 to 15 on one work-group (up to 2048 points) beside steps on slices (above)
    assert min(max(i for i, (_, s) in zip(its, bodies) if lo < s.N <= hi) for lo, hi in ((0, 2048), (2048, 4096))) > 9
    for k, (g, s) in enumerate(bodies):
        f1, s1, it1 = ilhip.DirichletPoisson(cs[k]).solve_moving(fbs[k], tol=1e-12, max_iter=200)
        print("N", s.N, "GMRES steps", it1, flush=True)
        assert its[k] == it1 and it1 > 0
        assert np.array_equal(fd[k].download(), f1.flat()) and np.array_equal(sd[k].download(), s1.flat())
        fr, _ = ilhip.DirichletPoisson(ilhip.SurfaceScalarCache(moved[k], g, ctx=ctx)).solve(fbs[k], filter_power=0)
        assert rel_err(f1.flat(), fr.flat()) < 1e-10
