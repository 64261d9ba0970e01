"""The Morton order over the sizes at which the radix sort changes its tiles."""
import numpy as np
import pytest

from timothy_amd import generators as gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(tm):
    c = tm.Context(0)
    yield c
    c.close()


def morton(x, y, z, ext):
    """87-bit keys (level 28 first, z, y, x within a level), as two words"""
    lo = [v.min() - ext for v in (x, y, z)]
    hi = [v.max() + ext for v in (x, y, z)]
    side = max(h - l for h, l in zip(hi, lo))
    code = [(((v - l) / side) * 536870912.0).astype(np.uint64) for v, l in zip((x, y, z), lo)]
    words = [np.zeros(x.size, np.uint64), np.zeros(x.size, np.uint64)]
    for bit in range(28, -1, -1):
        w = 0 if bit >= 14 else 1
        for c in (code[2], code[1], code[0]):
            words[w] = (words[w] << np.uint64(1)) | ((c >> np.uint64(bit)) & np.uint64(1))
    return words


# one workgroup's sort, a tile's edges, the last and first size of each rule
@pytest.mark.parametrize("n", [2, 63, 1025, 2048, 2049, 4095, 4096, 4097, 16 * 1024 + 1, 65536, 65537, 786432, 786433, 4194304, 4194305])
def test_order_is_morton_order(tm, ctx, n):
    pos = np.random.default_rng(n).random((n, 3)) * max(n, 1000) ** (1 / 3)
    col = gen._cells(pos, np.zeros(n, np.int32), gen.Stream(7, 2), gen.CELLTYPES)
    print(f"order of {n} cells", flush=True)
    ctx.upload_colony(col)
    ctx.build()
    hi, lo = morton(*pos.T, gen.CELLTYPES[0]["h"] + 0.01)
    perm, _ = ctx.order()
    assert np.array_equal(perm, np.lexsort((lo, hi)))
