"""A captured graph holds the addresses of the context's memory and the sizes of its cells:
calls that free any of it or change them retire the graph (a launch then fails until the next
capture), others leave it."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


def colony(n, h, seed=5):
    col = gen.ball_colony(n, seed)
    col["types"] = [dict(size=1.0, h=h, h2=h * h, h3=h ** 3, h4=h ** 4)]
    return col


def more_cells(tm, ctx):
    ctx.upload_colony(colony(4000, 2.0))


def a_few_more_cells(tm, ctx):
    ctx.upload_colony(colony(2100, 2.0))  # within the cell arrays' room


def fewer_cells(tm, ctx):
    ctx.upload_colony(colony(1900, 2.0))


def more_colonies(tm, ctx):
    ctx.upload_colonies([colony(20, 2.0, s) for s in range(100)])


def longer_lists(tm, ctx):
    ctx.upload_colony(colony(2000, 6.0))
    ctx.step(tm.FP64)


def larger_tiles(tm, ctx):
    ctx.autotune(tm.MIXED)


@pytest.mark.parametrize("call", [more_cells, a_few_more_cells, fewer_cells, more_colonies, longer_lists, larger_tiles],
                         ids=lambda f: f.__name__)
def test_retired_with_its_memory(tm, call):
    with tm.Context(0) as ctx:
        ctx.upload_colony(colony(2000, 2.0))
        ctx.set_param("nbr_cap", 16)
        ctx.graph_capture(tm.MIXED)
        ctx.graph_launch()
        call(tm, ctx)
        with pytest.raises(tm.TMError) as e:
            ctx.graph_launch()
        assert e.value.status == 5  # TM_ERR_STATE: no captured graph
        ctx.graph_capture(tm.MIXED)
        ctx.step(tm.MIXED)
        ref = ctx.results()
        ctx.graph_launch()
        got = ctx.results()
        assert all(np.array_equal(got[k], ref[k]) for k in ref)


def test_kept_through_other_calls(tm):
    """the same cells again, sums in the other form, a transfer, a solve and the octree"""
    col = colony(2000, 2.0)
    with tm.Context(0) as ctx:
        ctx.upload_colony(col)
        ctx.graph_capture(tm.FP64)
        ctx.graph_launch()
        ref = ctx.results()
        pos = np.stack([col[k] for k in "xyz"])
        for nodes in (16, 40):  # the second in more memory
            grid = dict(lower=pos.min(axis=1), resolution=np.float32((pos.max() - pos.min()) / (nodes - 2)),
                        loweridx=np.zeros(3, int), upperidx=np.full(3, nodes - 1), localsize=np.full(3, nodes))
            f = tm.DeviceArray.from_host(ctx, np.full(nodes ** 3, 0.1))
            ctx.upload_colony(col)
            ctx.step(tm.MIXED)
            ctx.cic_deposit(grid, f)
            ctx.diffusion_step(grid, tm.Diffusion.make(0.1, 1.0), f)
            ctx.octree(0)
            ctx.graph_launch()
            got = ctx.results()
            assert all(np.array_equal(got[k], ref[k]) for k in ref)
            f.free()
