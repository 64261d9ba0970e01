"""The LDS tiles of the neighbour lists: what the context reports of them, and the FP64
sums over them, which tm_neighbors and tm_sph take and a step does not."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def reported(ctx):
    return ctx.get_param("tile_lds"), ctx.get_param("tiles_over")


def test_reports_of_lists_without_tiles(tm, ctx):
    """0 records and 0 over-full tiles where the lists have none: made with sph_tiles off
    after lists that had some, also once it is on again, and in 2-D, where no sum reads
    tiles; after an FP64 step those that a further sum would make, as tm_neighbors does"""
    col = gen.ball_colony(6000, 99)
    h = 7.0  # more distinct neighbours than a tile holds
    col["types"] = [dict(size=1.0, h=h, h2=h * h, h3=h ** 3, h4=h ** 4)]
    ctx.upload_colony(col)
    ctx.build()
    ctx.neighbors()
    lds, over = reported(ctx)
    assert lds > 0 and over > 0
    ctx.step(tm.FP64)
    assert reported(ctx) == (lds, over)
    try:
        ctx.set_param("sph_tiles", 0)
        ctx.neighbors()
        assert reported(ctx) == (0, 0)
        ctx.step(tm.FP64)
        assert reported(ctx) == (0, 0)
        ctx.set_param("sph_tiles", 1)
        assert reported(ctx) == (0, 0)
        ctx.step(tm.MIXED)
        assert reported(ctx) == (lds, over)
    finally:
        ctx.set_param("sph_tiles", 1)
    flat = dict(gen.ball_colony(3000, 9), z=np.zeros(3000), dimension=2)
    ctx.upload_colony(flat)
    ctx.step(tm.FP64)
    assert reported(ctx) == (0, 0)
    ctx.sph(tm.MIXED)
    assert reported(ctx) == (0, 0)
    ctx.set_celltypes(gen.CELLTYPES, 3)


def ball(n, seed, h):
    col = gen.ball_colony(n, seed)
    col["types"] = [dict(size=1.0, h=h, h2=h * h, h3=h ** 3, h4=h ** 4)]
    return col


# a few tiles beyond four workgroups' share of LDS (their records come from memory with
# the cap), tiles near the hash set's limit, more distinct neighbours than a tile holds
@pytest.mark.parametrize("make,staged,width", [
    (lambda: gen.config(4, scale=0.04), {0: (1281, 1537), 1: (1280, 1280)}, 256),
    (lambda: ball(40000, 5, 5.4), {0: (1281, 1537), 1: (1281, 1537)}, 256),
    (lambda: ball(6000, 99, 7.0), {0: (1537, 1537), 1: (1537, 1537)}, 256),
    (lambda: ball(40000, 5, 5.4), {0: (513, 1537), 1: (513, 1537)}, 512),
    (lambda: ball(40000, 5, 5.4), {0: (513, 1537), 1: (513, 1537)}, 128)],
    ids=["2M two types", "40K", "6K", "40K, 512 a tile", "40K, 128 a tile"])
def test_fp64_sums_over_tiles(tm, ctx, make, staged, width):
    """capped and uncapped, with the bitmap and with the hash set alone: the bits of a
    step's sums, which are taken from the lists"""
    ctx.upload_colony(make())
    ctx.set_param("tile_width", width)
    try:
        ctx.step(tm.FP64)
        ref = ctx.results()
        for cap in (0, 1):
            for window in (0, 1):
                ctx.set_param("tile_cap4", cap)
                ctx.set_param("tile_window", window)
                ctx.build()
                ctx.neighbors()  # with tiles
                ctx.sph(tm.FP64)
                got = ctx.results()
                lds, over = reported(ctx)
                print(f"cap {cap}, window {window}: {lds} records staged, {over} over-full tiles", flush=True)
                assert staged[cap][0] <= lds <= staged[cap][1]
                assert all(np.array_equal(got[k], ref[k]) for k in ref)
    finally:
        for k, v in (("tile_cap4", 1), ("tile_window", 1), ("tile_width", 256)):
            ctx.set_param(k, v)
