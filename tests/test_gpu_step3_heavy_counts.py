"""Heavy rows in numbers around the 128 that their blocks are laid out in."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 15, 16, 17, 127, 128, 129, 200, 256, 300])
def test_any_number_of_heavy_rows(ctx, count):
    rng = np.random.default_rng(count)
    n, rows = 7000, 400  # seven parts of 1024 columns
    b = ts.gen_er(n, 9.0, seed=2)
    per = np.full(rows, 3)
    per[rng.choice(rows, count, replace=False)] = 150  # 1350 products or so, the others 27
    cols = [np.sort(rng.choice(n, k, replace=False)) for k in per]
    a = ts.Csr(rows, n, np.r_[0, np.cumsum(per)], np.concatenate(cols), rng.uniform(-1, 1, int(per.sum())))
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    tune = ts.default_tune()
    tune.force_tile_parallel = 1
    plain, _ = ctx.spgemm(ta, tb, tune)
    want = ctx.download_tiles(plain)
    ctx.build_rowindex(ta)
    ctx.build_rowindex(tb)
    tune = ts.default_tune()
    tune.element_mode = 2
    tune.heavy_min_products = 700
    c, st = ctx.spgemm(ta, tb, tune)
    log(f"[heavy] {st.heavy_rows} rows")
    assert st.heavy_rows == count
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
        assert np.array_equal(got[k], want[k]), k
    for x in (plain, c, ta, tb, da, db):
        ctx.free(x)
