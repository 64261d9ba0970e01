"""The environment solve over grid shapes at the edges of its kernels' tiles and of
the rule between them, against the oracle's solution."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def grid_of(ls, res):
    return dict(lower=[0.0] * 3, resolution=np.float32(res), loweridx=[0, 0, 0],
                upperidx=[int(v) - 1 for v in ls], localsize=[int(v) for v in ls])


@pytest.mark.parametrize("ls", [(1, 1, 1), (3, 1, 1), (1, 5, 1), (2, 1, 7), (16, 16, 20), (17, 17, 18), (8, 10, 128),
                                (11, 7, 133), (7, 9, 257), (33, 8, 128), (5, 63, 65), (1, 130, 129), (130, 1, 129),
                                (4, 32776, 2), (40, 65, 8), (31, 70, 5), (30, 40, 16), (15, 35, 31), (11, 31, 32)])
def test_diffusion_grid_shapes(tm, oracle_mod, ctx, ls):
    """axes of one node, one workgroup's grids and the first past them (5,120 and 10,240
    nodes), partial tiles and runs, every tile shape, more tiles than workgroups: the oracle's solution,
    over one step and two and where the iterations run out.  Both sides stop at residuals
    of 1e-12 |b| <= 1e-12 (1 + 12 z) |u|, and the operator's least eigenvalue is above one:
    2 steps, 2 sides, z = 0.7: 4e-11 |u|"""
    O = oracle_mod
    res, dt, lam = 2.0, 16000.0, 0.01 / 16000.0
    D = 0.7 * 4.0 / dt
    rng = np.random.default_rng(ls[0] + 7 * ls[1] + 31 * ls[2])
    u0 = 0.1575 + 0.01 * rng.random(ls)
    src = 1e-2 * rng.random(ls)
    p = dict(diffusion=D, boundary=0.1575, dt=dt, **{"lambda": lam})
    say(f"diffusion grid {ls}")
    f = tm.DeviceArray.from_host(ctx, u0.ravel())
    s = tm.DeviceArray.from_host(ctx, src.ravel())
    for substeps, maxiter in ((1, 200), (2, 200), (1, 2)):
        f.set(u0.ravel())
        it, rel = ctx.diffusion_step(grid_of(ls, res), tm.Diffusion.make(D, dt, 0.1575, lam, 1e-12, maxiter, substeps),
                                     f, s)
        got = f.get()
        ref, it_ref = O.diffusion_solve(ls, res, p, u0, src, tol=1e-12, maxiter=maxiter, substeps=substeps)
        assert abs(it - it_ref) <= substeps and (rel <= 1e-12 or it == maxiter)
        assert np.linalg.norm(got - ref) <= 4e-11 * np.linalg.norm(ref)
    f.free()
    s.free()


# long grids of thin planes, taken with a lane per node: few and many planes, rows across
# workgroups, several nodes a lane (beyond 524,288); planes that fill just less than half
# the lanes of the march's blocks, and half; the march with more tiles than workgroups
@pytest.mark.parametrize("ls", [(5121, 2, 1), (2561, 2, 2), (1153, 3, 3), (5000, 3, 2), (160, 5, 13), (45, 15, 16),
                                (45, 16, 16), (81, 33, 33), (19, 9, 65), (60001, 3, 3), (262145, 2, 1), (131073, 2, 2),
                                (1, 1500, 1500)])
def test_diffusion_thin_planes(tm, oracle_mod, ctx, ls):
    """as above, with the same bound"""
    test_diffusion_grid_shapes(tm, oracle_mod, ctx, ls)


def test_diffusion_thin_planes_take_no_longer(tm, ctx):
    """a solve of two iterations on 100,000 x 3 x 3 nodes against one on as many in a
    cube: about its time with a lane per node, 8 times it in blocks of mostly idle lanes"""
    import time

    best = {}
    for ls in ((100000, 3, 3), (96, 96, 98)):
        u0 = np.full(int(np.prod(ls)), 0.15)
        f = tm.DeviceArray.from_host(ctx, u0)
        par = tm.Diffusion.make(1.8e-5 * 4.0, 1.0, 0.1575, 0.0, 1e-12, 400, 1)
        ts = []
        for _ in range(12):
            f.set(u0)
            ctx.sync()
            t0 = time.perf_counter()
            it, _rel = ctx.diffusion_step(grid_of(ls, 2.0), par, f)
            ts.append(time.perf_counter() - t0)
        say(f"{ls}: {it} iterations, {1e6 * min(ts):.0f} us")
        best[ls] = min(ts)
        f.free()
    assert best[(100000, 3, 3)] <= 3.0 * best[(96, 96, 98)]
