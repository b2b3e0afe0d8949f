"""Which tile-rows of a large product are taken row by row: those whose rows
have products enough for each group of column parts, not those whose products
are spread over many groups.  stats.heavy_bytes is that path's memory, 0 when
no row takes it."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def random_tiles(tile_rows, tiles, entries, seed=0):
    """`tiles` tiles of `entries` entries in each tile-row, anywhere."""
    rng = np.random.default_rng(seed)
    n = 16 * tile_rows
    key = np.unique(np.repeat(np.arange(tile_rows), tiles) * tile_rows + rng.integers(0, tile_rows, tile_rows * tiles))
    i, j = key // tile_rows, key % tile_rows
    at = np.argsort(rng.random((len(key), 256)), axis=1)[:, :entries]
    key = np.sort(((i[:, None] * 16 + at // 16) * n + j[:, None] * 16 + at % 16).ravel())
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return ts.Csr(n, n, ptr, key % n, rng.uniform(-1, 1, len(key)))


@pytest.mark.parametrize("name,a,by_rows", [
    ("48 products a group", lambda: random_tiles(3000, 8, 48), False),   # 575 a row over 12 groups
    ("48 products a group, small tiles", lambda: random_tiles(3000, 24, 16), False),  # 573 over 12
    ("390 products a group", lambda: random_tiles(1500, 24, 32), True),  # 2270 over 6
    ("400 products a group", lambda: ts.gen_er(16384, 40.0, seed=1), True),
], ids=["48", "48_small_tiles", "390", "400_er"])
def test_rows_with_few_products_a_group_stay_in_segments(ctx, name, a, by_rows):
    a = a()
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    ctx.build_csc(t)
    ctx.build_rowindex(t)
    c, st = ctx.spgemm(t, t)
    log(f"[long rule] {name}: C {st.nnzC}, row path's bytes {st.heavy_bytes}")
    assert st.nnzC >= 12 << 20  # from here on tile-rows may go row by row
    assert (st.heavy_bytes > 0) == by_rows
    got = ctx.checksum(c).key()
    ctx.free(c)
    tune = ts.default_tune()
    tune.no_heavy_rows = 1
    c, _ = ctx.spgemm(t, t, tune)
    assert ctx.checksum(c).key() == got
    for x in (c, t, d):
        ctx.free(x)
