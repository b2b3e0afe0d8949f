"""Heavy rows against a B of few rows and more than 2^26 columns: more windows
of 1024 columns than a launch has grid rows."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1 << 26, (1 << 26) + 1040, (1 << 27) - 32])
def test_heavy_rows_of_a_wide_b(ctx, n):
    rng = np.random.default_rng(n % 97)
    rows = 260
    cols = [np.unique(np.r_[0, n - 1, rng.integers(0, n, 40), rng.integers(0, 3000, 60)]) for _ in range(rows)]
    b = ts.Csr(rows, n, np.r_[0, np.cumsum([len(c) for c in cols])], np.concatenate(cols),
               rng.uniform(-1, 1, sum(len(c) for c in cols)))
    pick = [np.sort(rng.choice(rows, k, replace=False)) for k in [200, 3, 0, 150, 1] + [2] * 30]
    a = ts.Csr(len(pick), rows, np.r_[0, np.cumsum([len(c) for c in pick])], np.concatenate(pick),
               rng.uniform(-1, 1, sum(len(c) for c in pick)))
    log(f"[wide] B {rows} x {n} nnz {b.nnz}")
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
    tune.heavy_min_products = 5000
    c, st = ctx.spgemm(ta, tb, tune)
    assert st.heavy_rows == 2
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
        assert np.array_equal(got[k], want[k]), k
    for x in (plain, c, ta, tb, da, db):
        ctx.free(x)
