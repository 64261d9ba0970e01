"""The LDS tiles of the neighbour lists: what the context reports of them."""
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
