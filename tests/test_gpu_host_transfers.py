"""Uploads and results through pinned memory and by direct copies: the cells that arrive
are the last uploaded, whatever the sizes, the optional arrays and what is in flight."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def colony(n, seed):
    col = gen.ball_colony(n, seed)
    rng = np.random.default_rng(seed)
    col["phase"] = rng.integers(0, 3, n).astype(np.int32)
    col["young"] = rng.random(n).astype(np.float32)
    return col


# around the padding, and around the sizes at which results (87,381 cells) and inputs
# (95,325) no longer go through pinned memory
@pytest.mark.parametrize("n", [2, 63, 64, 65, 3000, 87381, 87382, 95296, 95400])
@pytest.mark.parametrize("optional", [True, False])
def test_last_upload_is_what_a_step_sees(tm, ctx, n, optional):
    print(f"uploads of {n} cells, optional arrays {optional}", flush=True)
    a, b, c = colony(n, 3), colony(n, 4), colony(max(2, n // 2), 5)
    ctx.set_celltypes(gen.CELLTYPES, 3)
    arrays = lambda q: [q[k] for k in ("x", "y", "z", "size")] + [q["young"] if optional else None, q["ctype"],
                                                                  q["phase"] if optional else None]
    for q in (c, a, b):  # each while the one before may still be copied
        host = [None if v is None else v.copy() for v in arrays(q)]
        ctx.upload(*host)
        for v in host:
            if v is not None:
                v.fill(0)  # the caller's arrays are free again
    ctx.step(tm.FP64)
    got, pos = ctx.results(), ctx.positions()
    assert all(np.array_equal(p, b[k]) for p, k in zip(pos, "xyz"))
    dev = [None if v is None else tm.DeviceArray.from_host(ctx, v) for v in arrays(b)]
    ctx.bind_device(n, *dev)
    ctx.step(tm.FP64)
    ref = ctx.results()
    # bit for bit (without Young's moduli v is no number)
    assert all(np.array_equal(got[k].view(np.uint64), ref[k].view(np.uint64)) for k in ref)
    for v in dev:
        if v is not None:
            v.free()


def test_results_of_some_arrays(tm, ctx):
    col = colony(500, 6)
    ctx.upload_colony(col)
    ctx.step(tm.FP64)
    ref = ctx.results()
    v = np.full(500, -1.0)
    ctx._check(tm.lib().tm_get_results(ctx.h, None, v.ctypes.data, None, None, None, None))
    assert np.array_equal(v, ref["v"])


# around the sizes from which two, one and no arrays between those asked for are copied
# with them, and at which results no longer go through pinned memory
@pytest.mark.parametrize("n", [2, 8192, 8193, 16384, 16385, 32768, 32769, 87381, 87382])
def test_results_of_any_arrays(tm, ctx, n):
    print(f"results of {n} cells", flush=True)
    ctx.upload_colony(colony(n, 7))
    ctx.step(tm.FP64)
    r = ctx.results()
    ref = [r["density"], r["v"], r["mindist"]] + [np.ascontiguousarray(r["force"][:, a]) for a in range(3)]
    for which in range(64):
        got = [np.full(n, -1.0) if which >> j & 1 else None for j in range(6)]
        ctx._check(tm.lib().tm_get_results(ctx.h, *[None if g is None else g.ctypes.data for g in got]))
        assert all(g is None or np.array_equal(g, q) for g, q in zip(got, ref)), which


def test_one_array_is_all_that_is_copied(tm, ctx):
    """one array at the last size that goes through pinned memory takes as long as at the
    first that does not (2.2 times that where all six were copied)"""
    import time

    best = {}
    for n in (87381, 87382):
        ctx.upload_colony(colony(n, 7))
        ctx.step(tm.FP64)
        v, ts = np.empty(n), []
        for _ in range(60):
            t0 = time.perf_counter()
            ctx._check(tm.lib().tm_get_results(ctx.h, None, v.ctypes.data, None, None, None, None))
            ts.append(time.perf_counter() - t0)
        best[n] = min(ts)
        print(f"one array of {n} cells: {1e6 * best[n]:.0f} us", flush=True)
    assert best[87381] <= 1.5 * best[87382]
