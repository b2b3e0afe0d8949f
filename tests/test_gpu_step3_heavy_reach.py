"""Heavy and long rows whose tile-rows reach a few of B's column parts, some of
them many: a row has blocks by what the rows reach on average, and takes
several of its parts a block where it reaches more."""
import time

import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def near_diagonal(rows, n, half, per, wide, wide_per, seed):
    """`per` entries a row within `half` of the diagonal (row i at column i * n
    / rows); the rows of the tile-rows `wide` have `wide_per` anywhere."""
    rng = np.random.default_rng(seed)
    cols = []
    for i in range(rows):
        if i // 16 in wide:
            cols.append(np.sort(rng.choice(n, wide_per, replace=False)))
        else:
            lo = min(max(i * n // rows - half, 0), n - 2 * half)
            cols.append(lo + np.sort(rng.choice(2 * half, per, replace=False)))
    ptr = np.r_[0, np.cumsum([len(c) for c in cols])]
    return ts.Csr(rows, n, ptr, np.concatenate(cols), rng.uniform(-1, 1, int(ptr[-1])))


@pytest.mark.parametrize("heavy", [False, True], ids=["long", "heavy"])
@pytest.mark.parametrize("rows", [112, 128, 1008, 1024, 1040, 2176])
def test_rows_that_reach_more_parts_than_the_others(ctx, rows, heavy):
    n = 61000  # 60 parts, 15 groups
    b = near_diagonal(n, n, 700, 24, (), 0, 1)
    a = near_diagonal(rows, n, 900, 40, (2, 5), 130, 2)  # 960 products a row, 3120 of the wide ones
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
    tune.heavy_min_products = 700 if heavy else 1 << 30
    c, st = ctx.spgemm(ta, tb, tune)
    log(f"[reach] {rows} rows, {st.heavy_rows} heavy, bytes {st.heavy_bytes}")
    assert st.heavy_rows > 0.9 * rows if heavy else st.heavy_bytes > 0
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
        assert np.array_equal(got[k], want[k]), k
    for x in (plain, c, ta, tb, da, db):
        ctx.free(x)


def test_wide_band_costs_what_its_rows_reach(ctx):
    """1,000,000 rows that reach 8 of 977 parts: not a wave per row and part
    (6.5 times the time by segments alone; the bound is 3)."""
    n, half, per = 1000000, 2000, 24
    rng = np.random.default_rng(3)
    i = np.repeat(np.arange(n), per)
    key = np.unique(i * n + np.clip(i + rng.integers(-half, half + 1, n * per), 0, n - 1))
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    d = ctx.upload(ts.Csr(n, n, ptr, key % n, rng.uniform(-1, 1, len(key))))
    t = ctx.csr2tile(d)
    ctx.build_csc(t)
    ctx.build_rowindex(t)
    best, sums = [], []
    for segments in (0, 1):
        tune = ts.default_tune()
        tune.no_heavy_rows = segments
        times = []
        for _ in range(4):
            ctx.sync()
            t0 = time.perf_counter()
            c, _ = ctx.spgemm(t, t, tune, timed=False)
            ctx.sync()
            times.append(time.perf_counter() - t0)
            if len(times) == 1:
                sums.append(ctx.checksum(c).key())
            ctx.free(c)
        best.append(min(times))
    log(f"[reach] {best[0] * 1e3:.2f} ms, by segments {best[1] * 1e3:.2f}")
    assert sums[0] == sums[1]
    assert best[0] < 3 * best[1]
    for x in (t, d):
        ctx.free(x)
