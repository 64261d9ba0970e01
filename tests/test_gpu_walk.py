"""The cooperative walk (walk_coop, one walk per wave) against the per-lane
walk of the radix tree: lists, last candidates, mindist, v and the FP64 sums
equal bit for bit, at the sizes where its cells per wave and the levels of its
tree of boxes change, and on colonies that take its rarer branches -- cells in
many places, cells without a neighbour beside crowded ones, queues longer than
their room, waves of many small colonies."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def gaussian(n):
    return gen.gaussian_colony(n, 900 + n % 89, 146.6 * (n / 2e6) ** (1 / 3), frac_type1=0.05)


def cells(pos, types=gen.CELLTYPES):
    n = len(pos)
    return gen._cells(np.asarray(pos, np.float64), np.zeros(n, np.int32), gen.Stream(7, 2), types)


def wide_type(h):
    return [dict(size=1.0, h=h, h2=h ** 2, h3=h ** 3, h4=h ** 4)]


def scattered(n):
    """far apart: no cell has a neighbour"""
    return cells(gen.Stream(31, 1).uniform(3 * n).reshape(n, 3) * 4000.0)


def crowd_and_strays(n):
    """a dense ball and lone cells around it, a cutoff of seven radii: waves
    with hundreds of candidates hold cells without a neighbour"""
    st = gen.Stream(33, 1)
    ball = gen.uniform_ball(n, 0.9 * n ** (1 / 3), st)
    out = gen.uniform_ball(400, 60.0 * n ** (1 / 3) / 10, st)
    out = out[(out ** 2).sum(1) > (0.9 * n ** (1 / 3) + 8) ** 2]
    return cells(np.concatenate([ball, out]), wide_type(7.0))


def clusters(k, m):
    """k small clumps far apart, in an order that mixes them within waves"""
    st = gen.Stream(35, 1)
    at = st.uniform(3 * k).reshape(k, 3) * 900.0
    return cells((at[:, None, :] + gen.Stream(36, 1).normal(3 * k * m).reshape(k, m, 3)).reshape(-1, 3))


CASES = [(f"gaussian {n}", lambda n=n: gaussian(n))
         for n in (2, 15, 63, 65, 1023, 1025, 32768, 32769, 65537, 131073)] + [
    ("scattered", lambda: scattered(5000)),
    ("crowd and strays", lambda: crowd_and_strays(6000)),
    ("clusters", lambda: clusters(700, 5)),
    ("far cutoff", lambda: dict(gen.ball_colony(9000, 41), types=wide_type(9.0))),
]


def outputs(tm, ctx, coop, lists):
    ctx.set_param("walk_coop", coop)
    ctx.step(tm.FP64)
    return dict(ctx.results(), qstar=ctx.qstar(), **(dict(zip(("off", "nbr"), ctx.neighbor_lists())) if lists else {}))


@pytest.mark.parametrize("name,make", CASES)
@pytest.mark.parametrize("ratio", [64, 3])
def test_matches_per_lane_walk(tm, ctx, name, make, ratio):
    ctx.upload_colony(make())
    ctx.set_param("walk_coop_ratio", ratio)
    ref, got = outputs(tm, ctx, 0, True), outputs(tm, ctx, 1, True)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k
    ctx.set_param("walk_coop_ratio", 64)


def test_small_colonies_in_one_wave(tm, ctx):
    cols = [gaussian(m) for m in [1, 2, 3, 5, 8, 13, 21, 34, 55, 89, 144, 233] * 30]
    ctx.upload_colonies(cols)
    ref, got = outputs(tm, ctx, 0, True), outputs(tm, ctx, 1, True)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("n", [786433, 4194305 + 70])
def test_matches_per_lane_walk_large(tm, ctx, n):
    ctx.upload_colony(gaussian(n))
    ref, got = outputs(tm, ctx, 0, False), outputs(tm, ctx, 1, False)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


def test_octree_on_demand(tm, ctx):
    """the radix tree is made when asked for: after a cooperative step, and
    anew after a replay of a captured one"""
    ctx.upload_colony(gaussian(3000))
    ctx.set_param("walk_coop", 0)
    ctx.step(tm.MIXED)
    ref = ctx.octree(0)
    ctx.set_param("walk_coop", 1)
    ctx.graph_capture(tm.MIXED)
    for _ in range(3):
        ctx.graph_launch()
        assert np.array_equal(ctx.octree(0), ref)
    ctx.graph_destroy()


def test_fp64_sums_with_and_without_tiles(tm, ctx):
    """a step's one FP64 sum is taken from the lists, later sums over tiles:
    the same bits; a mixed sum after it is the one of a mixed step; tiles of a
    replay's lists are not those of the lists before"""
    ctx.upload_colony(gaussian(20011))
    ctx.step(tm.MIXED)
    mixed = ctx.results()
    ctx.step(tm.FP64)
    first = ctx.results()
    for _ in range(10):
        ctx.sph(tm.FP64)
    over_tiles = ctx.results()
    ctx.sph(tm.MIXED)
    again = ctx.results()
    for k in first:
        assert np.array_equal(over_tiles[k], first[k]) and np.array_equal(again[k], mixed[k]), k
    ctx.graph_capture_loop(tm.Move.make([0.2, 0.2], seed=5), tm.FP64)
    for _ in range(2):
        ctx.sph(tm.MIXED)
        ctx.graph_launch()
        got = ctx.results()
        ctx.sph(tm.MIXED)
        ctx.sph(tm.FP64)
        for k in got:
            assert np.array_equal(ctx.results()[k], got[k]), k
    ctx.graph_destroy()


def sparse(n, fraction, seed=51, shift=0.0, scale=1.0):
    """a ball with `fraction` of its volume in cells: 0.08 leaves 53 % without a neighbour"""
    p = gen.uniform_ball(n, (n / fraction) ** (1 / 3), gen.Stream(seed, 1)) * scale + shift
    return cells(p, [dict(size=scale, h=2 * scale, h2=4 * scale ** 2, h3=8 * scale ** 3, h4=16 * scale ** 4)])


# 32 and 64 cells a wave; from a few to all of a wave's cells without a neighbour, beside
# some candidates and beside more than are kept; far from the origin; squares beyond FP32
@pytest.mark.parametrize("name,make", [
    ("32, 0.3", lambda: sparse(140001, 0.3)), ("32, 0.15", lambda: sparse(140011, 0.15)),
    ("32, 0.05", lambda: sparse(300007, 0.05)), ("32, 0.005", lambda: sparse(140003, 0.005)),
    ("64, 0.3", lambda: sparse(800011, 0.3)), ("64, 0.12", lambda: sparse(800029, 0.12)),
    ("64, 0.04", lambda: sparse(800033, 0.04)), ("64, 0.005", lambda: sparse(790001, 0.005)),
    ("scattered", lambda: scattered(200003)), ("far", lambda: sparse(150001, 0.06, shift=1e6)),
    ("beyond FP32", lambda: sparse(140009, 0.06, scale=3e17)),
    ("two cutoffs", lambda: dict(sparse(200001, 0.1), ctype=(np.arange(200001) % 3 == 0).astype(np.int32),
                                 types=[wide_type(1.1)[0], wide_type(2.3)[0]]))])
def test_cells_without_a_neighbour(tm, ctx, name, make):
    ctx.upload_colony(make())
    ref, got = outputs(tm, ctx, 0, True), outputs(tm, ctx, 1, True)
    alone = float(np.mean(np.diff(ref["off"]) == 0))
    print(f"{name}: {100 * alone:.0f} % without a neighbour", flush=True)
    assert alone > 0.05
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


def test_cells_without_a_neighbour_of_many_colonies(tm, ctx):
    cols = [sparse(40 + 97 * (i % 9), (0.3, 0.08, 0.01)[i % 3], seed=60 + i % 9) for i in range(900)]
    ctx.upload_colonies(cols)
    ref, got = outputs(tm, ctx, 0, True), outputs(tm, ctx, 1, True)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


def test_sparse_colony_takes_no_longer(tm, ctx):
    """a step of 1M cells, three quarters of them without a neighbour, takes about as long as
    with one lane per cell (0.95 times that; 1.7 times where they went two or one at a time)"""
    import time

    ctx.upload_colony(sparse(1000000, 0.04))
    best = {}
    for coop in (0, 1):
        ctx.set_param("walk_coop", coop)
        ts = []
        for _ in range(12):
            ctx.sync()
            t0 = time.perf_counter()
            ctx.step(tm.FP64)
            ctx.sync()
            ts.append(time.perf_counter() - t0)
        best[coop] = min(ts)
    print(f"one lane per cell {1e6 * best[0]:.0f} us, together {1e6 * best[1]:.0f} us", flush=True)
    assert best[1] <= 1.3 * best[0]


# colonies at and past the mean size from which waves take their cells together, for each
# number of cells a wave
@pytest.mark.parametrize("m,size", [(1000, 4), (1000, 5), (5000, 8), (5000, 9), (9000, 16), (9000, 17), (30000, 28),
                                    (30000, 29)])
def test_many_small_colonies(tm, ctx, m, size):
    one = [gen.ball_colony(size, 70 + i) for i in range(30)]
    ctx.upload_colonies([one[i % 30] for i in range(m)])
    ref, got = outputs(tm, ctx, 0, False), outputs(tm, ctx, 1, False)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k
    ctx.graph_capture(tm.FP64)
    for _ in range(2):
        ctx.graph_launch()
        again = ctx.results()
        assert all(np.array_equal(again[k], ref[k]) for k in again)
    ctx.graph_destroy()


def test_many_small_colonies_take_no_longer(tm, ctx):
    """a step of 50,000 colonies of three cells takes as long as with one lane per cell (1.5
    times that where a wave took five colonies one after another)"""
    import time

    one = [gen.ball_colony(3, 70 + i) for i in range(30)]
    ctx.upload_colonies([one[i % 30] for i in range(50000)])
    best = {}
    for coop in (0, 1):
        ctx.set_param("walk_coop", coop)
        ts = []
        for _ in range(12):
            ctx.sync()
            t0 = time.perf_counter()
            ctx.step(tm.FP64)
            ctx.sync()
            ts.append(time.perf_counter() - t0)
        best[coop] = min(ts)
    print(f"one lane per cell {1e6 * best[0]:.0f} us, by default {1e6 * best[1]:.0f} us", flush=True)
    assert best[1] <= 1.2 * best[0]
