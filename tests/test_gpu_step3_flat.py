"""Numeric step of element-wise tile-rows with both row indices: segment
edges (one segment, one more nonzero, many), rows of very different lengths,
sources that meet in one C entry inside a batch and across batches, heavy rows
beside light ones, spans past the packed hash keys, ragged last tile-rows,
infinities and NaN.  Values are compared with the tile-pair path bit for bit
(its own order is the oracle's, checked on one case here)."""
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


def inputs():
    rng = np.random.default_rng(7)

    def some(n, k):
        return np.sort(rng.choice(n, min(n, k), replace=False))

    # one C tile-row of t nonzeros: A row 0 picks B rows with disjoint columns
    for t in (1, 64, 65, 255, 256, 257, 2240, 2241, 2242, 2496, 2497, 9000):
        a = {0: [0, 1, 2]}
        cols = np.arange(t) * 7
        b = {0: cols[0::3], 1: cols[1::3], 2: cols[2::3]}
        yield f"nnz{t}", csr(16, 3, a), csr(3, 7 * t + 1, b), False
    # every source meets the others: 70 B rows over the same 100 columns
    yield "same_columns", csr(33, 70, {r: some(70, 1 + 2 * r) for r in range(33)}), csr(70, 5000, {r: some(100, 90) * 50 for r in range(70)}), False
    # a long row with fifteen short ones; 130 sources (three batches of 64)
    a = {r: some(400, 2) for r in range(48)}
    a[3] = some(400, 130)
    a[40] = np.arange(400)
    yield "uneven", csr(48, 400, a), csr(400, 30000, {r: some(30000, 5 + r % 60) for r in range(400)}), False
    # full tiles (256 entries) and a ragged last tile-row
    yield "dense", csr(75, 90, {r: np.arange(90) for r in range(75)}), csr(90, 700, {r: np.arange(700) for r in range(90)}), False
    # 70001 tile columns: hash keys past 20 bits
    yield "wide", csr(20, 40, {r: some(40, 6) for r in range(20)}), csr(40, 16 * 70001, {r: np.unique(np.r_[0, some(16 * 70001, 300), 16 * 70001 - 1]) for r in range(40)}), False
    # heavy rows (more products than 65536, more than 2048 A entries) beside light ones
    a = {r: some(3000, 4) for r in range(40)}
    a[5] = np.arange(3000)
    a[6] = some(3000, 1500)
    yield "heavy", csr(40, 3000, a), csr(3000, 9000, {r: some(9000, 60) for r in range(3000)}), True
    a = {r: some(300, 250) for r in range(32)}
    yield "heavy_long_b", csr(32, 300, a), csr(300, 6000, {r: some(6000, 2500) for r in range(300)}), True


@pytest.mark.parametrize("name,a,b,heavy", list(inputs()), ids=[i[0] for i in inputs()])
@pytest.mark.parametrize("special", [False, True])
def test_flat_matches_tile_pairs(ctx, name, a, b, heavy, special):
    log(f"[step3 flat] {name} A {a.m}x{a.n} nnz {a.nnz} B {b.m}x{b.n} nnz {b.nnz} special {special}")
    if special:  # values that must not spread to entries they take no part in
        a = ts.Csr(a.m, a.n, a.rowptr, a.colidx, a.val.copy())
        b = ts.Csr(b.m, b.n, b.rowptr, b.colidx, b.val.copy())
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
    c, st = ctx.spgemm(ta, tb, tune)
    assert (st.heavy_rows > 0) == heavy
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask"):
        assert np.array_equal(got[k], want[k]), k
    assert np.array_equal(got["val"], want["val"], equal_nan=True)
    ok = ~np.isnan(want["val"])
    assert got["val"][ok].tobytes() == want["val"][ok].tobytes()
    # A without its row index: decoded from its tiles
    t2 = ctx.csr2tile(da)
    c2, _ = ctx.spgemm(t2, tb, tune)
    g2 = ctx.download_tiles(c2)
    assert np.array_equal(g2["val"], want["val"], equal_nan=True) and np.array_equal(g2["csr_col"], want["csr_col"])
    if name == "uneven" and not special:
        h = ctx.download(ctx.tile2csr(c))
        rp, cc, vc = oracle.spgemm(a, b)
        assert np.array_equal(h.rowptr.astype(np.int64), rp) and np.array_equal(h.colidx, cc) and np.array_equal(h.val, vc)
    for x in (c2, t2, c, plain, ta, tb, da, db):
        ctx.free(x)
