"""Numeric step of long and heavy rows: tile-rows of only such rows, runs of
column parts that fill the sums or stop short of it, sources that share C
entries, empty rows and rows without entries in some parts, ragged last
tile-rows and parts, windows wider than parts and a single window, infinities
and NaN.  Compared with the tile-pair path bit for bit (the oracle's order,
checked on one case here)."""
import numpy as np
import pytest

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def csr(m, n, rows, seed=1):
    ptr = np.zeros(m + 1, np.int64)
    for r, c in rows.items():
        ptr[r + 1] = len(c)
    cols = np.concatenate([np.asarray(rows[r], np.int32) for r in sorted(rows)] + [np.zeros(0, np.int32)])
    return ts.Csr(m, n, np.cumsum(ptr), cols, np.random.default_rng(seed).uniform(-1, 1, len(cols)))


def make(name):
    rng = np.random.default_rng(5)

    def some(n, k):
        return np.sort(rng.choice(n, min(n, k), replace=False))

    if name == "full_parts":  # every part full: runs of one part
        return csr(35, 6, {r: some(6, 1 + r % 5) for r in range(35)}), csr(6, 9001, {r: np.arange(r % 2, 9001) for r in range(6)})
    if name == "edge_1024":  # 1024, then 1025 entries in a run of two and of four parts
        a = {r: [r % 4] for r in range(16)}
        half, quarter = np.arange(0, 2048, 2), np.arange(0, 4096, 4)
        return csr(16, 4, a), csr(4, 5000, {0: half, 1: np.r_[half, 2047], 2: quarter, 3: np.r_[quarter, 4095]})
    if name == "few_long_sources":
        return csr(70, 40, {r: some(40, 2 + r % 9) for r in range(70) if r % 13}), csr(40, 20000, {r: some(20000, 1500 + 90 * r) for r in range(40)})
    if name == "many_short_sources":  # 64 and more sources a group, all over the same columns
        return csr(33, 900, {r: some(900, 60 + 20 * r) for r in range(33)}), csr(900, 6000, {r: some(300, 40) * 20 for r in range(900)})
    if name == "skewed":  # most entries in the first part, some rows only in the last
        b = {r: np.unique(np.r_[some(700, 300), some(30011, 40)]) for r in range(200)}
        b |= {r: 30011 - 1 - np.arange(100)[::-1] * 3 for r in range(0, 200, 9)}
        return csr(50, 200, {r: some(200, 20 + 3 * r) for r in range(50)}), csr(200, 30011, b)
    if name == "one_window":
        return csr(20, 300, {r: some(300, 250) for r in range(20)}), csr(300, 1024, {r: some(1024, 200) for r in range(300)})
    # the window table limited in size: windows of several parts
    m = 3000001
    return (csr(40, m, {r: some(3000, 30) * 1000 for r in range(40)}),
            csr(m, 100003, {1000 * r: some(100003, 400) for r in range(3000)}))


NAMES = ["full_parts", "edge_1024", "few_long_sources", "many_short_sources", "skewed", "one_window", "wide_windows"]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("least", [64, 1 << 30])  # rows above 64 products by single parts; every row by groups of parts
def test_long_rows_match_tile_pairs(ctx, name, least):
    a, b = make(name)
    log(f"[step3 long] {name} A {a.m}x{a.n} nnz {a.nnz} B {b.m}x{b.n} nnz {b.nnz} least {least}")
    for special in (False, True):
        if special:  # values that must not spread to entries they take no part in
            a.val[:: max(1, a.nnz // 5)] = np.inf
            b.val[:: max(1, b.nnz // 7)] = np.nan
            b.val[1 :: max(2, b.nnz // 3)] = -0.0
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
        tune.heavy_min_products = least
        c, _ = ctx.spgemm(ta, tb, tune)
        got = ctx.download_tiles(c)
        for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask"):
            assert np.array_equal(got[k], want[k]), k
        assert np.array_equal(got["val"], want["val"], equal_nan=True)
        ok = ~np.isnan(want["val"])
        assert got["val"][ok].tobytes() == want["val"][ok].tobytes()
        if name == "few_long_sources" and not special:
            h = ctx.download(ctx.tile2csr(c))
            rp, cc, vc = oracle.spgemm(a, b)
            assert np.array_equal(h.rowptr.astype(np.int64), rp) and np.array_equal(h.colidx, cc) and np.array_equal(h.val, vc)
        for x in (c, plain, ta, tb, da, db):
            ctx.free(x)
