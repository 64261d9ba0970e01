"""Field gradient and cloud-in-cell interpolation over grid shapes at the edges of
their kernels' waves, chunks and runs, in both types: bit-exact with the oracle."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def gradient_f32(f, res):
    g = np.empty(f.shape + (3,), np.float32)
    for a in range(3):
        F, E = np.moveaxis(f, a, 0), np.moveaxis(g[..., a], a, 0)
        E[1:-1] = (F[2:] - F[:-2]) / res
        E[0], E[-1] = (F[1] - F[0]) / res, (F[-1] - F[-2]) / res
    return g.reshape(-1)


# planes of less than a wave, a wave, more than a chunk of 256 columns; runs of planes that
# do not divide; beyond the L2 caches' size (the fewer workgroups of the interpolation)
@pytest.mark.parametrize("ls", [(2, 2, 2), (3, 7, 9), (9, 8, 8), (5, 5, 13), (33, 16, 16), (6, 17, 31), (2, 3, 341),
                                (13, 80, 81), (101, 103, 211)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_gradient_and_interp_grid_shapes(tm, oracle_mod, ctx, ls, dtype):
    O = oracle_mod
    col = gen.ball_colony(700, 5)
    pos = np.stack([col["x"], col["y"], col["z"]])
    # cells inside, on both faces and outside: the grid spans the middle of the colony
    res = np.float32(0.8 * (pos.max() - pos.min()) / min(ls))
    lower = pos.min(axis=1) + 0.1 * (pos.max() - pos.min())
    grid = dict(lower=lower, resolution=res, loweridx=np.array([0, -1, 1]), upperidx=np.array(ls) - 1 + [0, -1, 1],
                localsize=np.array(ls))
    total = int(np.prod(ls))
    f = np.random.default_rng(total).standard_normal(total).astype(dtype)
    ctx.upload_colony(col)
    ctx.build()
    f_d, g_d = tm.DeviceArray.from_host(ctx, f), tm.DeviceArray(ctx, 3 * total, dtype)
    out = tm.DeviceArray(ctx, 4 * col["n"], np.float64)
    print(f"transfers {ls} {np.dtype(dtype).name}", flush=True)
    ctx.field_gradient(grid, f_d, g_d)
    g = g_d.get()
    if dtype == np.float64:
        assert np.array_equal(g, O.fieldgradient(ls, res, f))
    else:
        assert np.array_equal(g, gradient_f32(f.reshape(ls), res))
    ctx.cic_interp(grid, f_d, g_d, out)
    ref = O.cic_interp(O.Colony.from_dict(col), grid, f.astype(np.float64), g.astype(np.float64))
    assert np.array_equal(out.get().reshape(-1, 4), ref)
    for a in (f_d, g_d, out):
        a.free()


@pytest.mark.parametrize("ls", [(64, 2, 2), (43, 3, 2), (300, 2, 3), (2, 2, 31), (9, 31, 2), (70, 7, 9), (70, 8, 8)])
def test_gradient_thin_planes(tm, oracle_mod, ctx, ls):
    """planes of less than 64 nodes, one lane a node: whole and partial workgroups, and the
    first plane past the rule; bit-exact in both types"""
    res = np.float32(1.7)
    grid = dict(lower=np.zeros(3), resolution=res, loweridx=np.zeros(3, int), upperidx=np.array(ls) - 1,
                localsize=np.array(ls))
    f = np.random.default_rng(int(np.prod(ls))).standard_normal(int(np.prod(ls)))
    for dtype in (np.float64, np.float32):
        print(f"thin gradient {ls} {np.dtype(dtype).name}", flush=True)
        v = f.astype(dtype)
        f_d, g_d = tm.DeviceArray.from_host(ctx, v), tm.DeviceArray(ctx, 3 * f.size, dtype)
        ctx.field_gradient(grid, f_d, g_d)
        want = oracle_mod.fieldgradient(ls, res, v) if dtype == np.float64 else gradient_f32(v.reshape(ls), res)
        assert np.array_equal(g_d.get(), want)


def gradient_of(f, res):
    """the kernels' expressions in f's type"""
    g = np.empty(f.shape + (3,), f.dtype)
    r = f.dtype.type(res)
    for a in range(3):
        F, E = np.moveaxis(f, a, 0), np.moveaxis(g[..., a], a, 0)
        E[1:-1] = (F[2:] - F[:-2]) / r
        E[0], E[-1] = (F[1] - F[0]) / r, (F[-1] - F[-2]) / r
    return g.reshape(-1)


# field and gradient of 32 and 192 MiB and the first sizes above: two and three planes,
# planes with partial chunks and waves, runs that do not divide; planes that fill three
# quarters of their chunks' lanes and less, up to 256 MiB and above
@pytest.mark.parametrize("ls,dtype", [
    ((64, 128, 128), np.float64), ((64, 128, 129), np.float64), ((2, 725, 726), np.float64),
    ((5449, 12, 16), np.float64), ((5449, 11, 17), np.float64), ((1031, 32, 33), np.float64),
    ((128, 128, 128), np.float32), ((128, 128, 129), np.float32), ((3, 841, 843), np.float32),
    ((8209, 15, 17), np.float32), ((11000, 10, 19), np.float32),
    ((96, 256, 256), np.float64), ((96, 256, 257), np.float64), ((3, 1459, 1460), np.float64),
    ((100003, 8, 8), np.float64), ((131073, 8, 8), np.float64), ((187, 185, 186), np.float64),
    ((32801, 12, 16), np.float64),
    ((192, 256, 256), np.float32), ((192, 257, 256), np.float32), ((235, 233, 234), np.float32),
    ((233021, 8, 9), np.float32), ((233025, 9, 8), np.float32)])
def test_gradient_by_size(tm, ctx, ls, dtype):
    """the three forms of the gradient on both sides of the lines between them: bit-exact"""
    res, n = np.float32(1.7), int(np.prod(ls))
    grid = dict(lower=np.zeros(3), resolution=res, loweridx=np.zeros(3, int), upperidx=np.array(ls) - 1,
                localsize=np.array(ls))
    print(f"gradient {ls} {np.dtype(dtype).name}", flush=True)
    v = np.random.default_rng(n).standard_normal(n).astype(dtype)
    f_d, g_d = tm.DeviceArray.from_host(ctx, v), tm.DeviceArray(ctx, 3 * n, dtype)
    ctx.field_gradient(grid, f_d, g_d)
    assert np.array_equal(g_d.get(), gradient_of(v.reshape(ls), res))
    f_d.free()
    g_d.free()


def test_sampling_finds_the_gradient_in_the_caches(tm, ctx):
    """gradient and interpolation of a small field one after the other take no longer than
    each repeated by itself (0.9 times that; 1.4 times where the gradient left past the
    caches)"""
    import time

    n, nodes = 1000000, 64
    col = gen.gaussian_colony(n, 3, 146.6 * (n / 2e6) ** (1 / 3))
    ctx.upload_colony(col)
    ctx.build()
    pos = np.stack([col[k] for k in "xyz"])
    res = np.float32((pos.max() - pos.min()) / (nodes - 2))
    grid = dict(lower=pos.min(axis=1), resolution=res, loweridx=np.zeros(3, int), upperidx=np.full(3, nodes - 1),
                localsize=np.full(3, nodes))
    f_d = tm.DeviceArray.from_host(ctx, np.random.default_rng(2).random(nodes ** 3).astype(np.float32))
    g_d, out = tm.DeviceArray(ctx, 3 * nodes ** 3, np.float32), tm.DeviceArray(ctx, 4 * n, np.float64)

    def gradient():
        ctx.field_gradient(grid, f_d, g_d)

    def interp():
        ctx.cic_interp(grid, f_d, g_d, out)

    def both():
        gradient()
        interp()

    def least(call):
        ts = []
        for _ in range(10):
            ctx.sync()
            t0 = time.perf_counter()
            for _ in range(40):
                call()
            ctx.sync()
            ts.append(1e6 * (time.perf_counter() - t0) / 40)
        return min(ts)

    both()
    g, i, b = least(gradient), least(interp), least(both)
    print(f"gradient {g:.1f} us, interpolation {i:.1f} us, both {b:.1f} us", flush=True)
    for a in (f_d, g_d, out):
        a.free()
    assert b <= 1.15 * (g + i)
