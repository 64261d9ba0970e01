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
