"""Numeric step by row lines (both row indices): the limits of C tiles and
nonzeros of a tile-row, the group sizes, A and B rows longer than a group,
tile-rows wider than the column map with and without columns that collide in
it, empty rows and ragged last tile-rows, runs of C at every alignment,
infinities and NaN.  Compared with the tile-pair path bit for bit (the
oracle's order, checked on two cases here)."""
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
    rng = np.random.default_rng(11)

    def some(n, k):
        return np.sort(rng.choice(n, min(n, k), replace=False))

    # C nonzeros of a tile-row: 16 rows of t, dense
    for t in (1, 2, 3, 5, 191, 192, 255, 256, 257):
        yield f"row{t}", csr(16, 1, {r: [0] for r in range(16)}), csr(1, t, {0: np.arange(t)})
    # C tiles of a tile-row
    for u in (255, 256, 257):
        yield f"tiles{u}", csr(17, 2, {r: [r & 1] for r in range(17)}), csr(2, 16 * u, {0: np.arange(0, 16 * u, 32), 1: np.arange(16, 16 * u, 32)})
    # B rows around the group sizes, two pieces a row, rows of uneven lengths
    for k in (1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129):
        yield f"brow{k}", csr(37, 50, {r: some(50, 20) for r in range(37)}), csr(50, 240, {r: some(240, k) for r in range(50)})
    for k in (31, 33, 80, 120, 150):
        yield f"uneven{k}", csr(40, 64, {r: some(64, 30) for r in range(40)}), csr(64, 200, {r: some(200, k if r % 9 == 0 else r % 25) for r in range(64)})
    # A rows of 0 to 200 entries beside each other; 2048 and 2049 in one tile-row
    for k in (2048, 2049):
        yield f"entries{k}", csr(16, 130, {r: some(130, 128 + (k - 2048 if r == 0 else 0)) for r in range(16)}), csr(130, 77, {r: some(77, 6) for r in range(130)})
    yield "long_a", csr(50, 200, {r: some(200, (r * 37) % 201) for r in range(50) if r % 7}), csr(200, 60, {r: some(60, 3 + r % 6) for r in range(200) if r % 11})
    # wide tile-rows: far columns that share a byte of the map, and that do not
    far = 16 * 8192
    yield "collide", csr(20, 30, {r: some(30, 9) for r in range(20)}), csr(30, 3 * far + 9, {r: np.unique(np.r_[some(64, 4), far + some(64, 4), 3 * far + 8 - some(8, 2)]) for r in range(30)})
    yield "wide", csr(20, 30, {r: some(30, 9) for r in range(20)}), csr(30, 3 * far + 9, {r: np.unique(np.r_[some(64, 4), far + 800 + some(64, 4), 3 * far - 900 + some(8, 2)]) for r in range(30)})
    # neighbouring tile-rows of different widths and group sizes
    yield "mixed", csr(16 * 9 + 5, 160, {r: 16 * (r // 16) + some(16, 1 + r % 7) for r in range(16 * 9 + 5)}), csr(160, 4000, {r: some(40 * (r // 16 + 1), 1 + 6 * (r // 16)) for r in range(160)})


@pytest.mark.parametrize("name,a,b", list(inputs()), ids=[i[0] for i in inputs()])
@pytest.mark.parametrize("special", [False, True])
def test_lines_match_tile_pairs(ctx, name, a, b, special):
    log(f"[step3 lines] {name} A {a.m}x{a.n} nnz {a.nnz} B {b.m}x{b.n} nnz {b.nnz} special {special}")
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
    c, _ = ctx.spgemm(ta, tb)
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask"):
        assert np.array_equal(got[k], want[k]), k
    assert np.array_equal(got["val"], want["val"], equal_nan=True)
    ok = ~np.isnan(want["val"])
    assert got["val"][ok].tobytes() == want["val"][ok].tobytes()
    if name in ("mixed", "long_a") and not special:
        h = ctx.download(ctx.tile2csr(c))
        rp, cc, vc = oracle.spgemm(a, b)
        assert np.array_equal(h.rowptr.astype(np.int64), rp) and np.array_equal(h.colidx, cc) and np.array_equal(h.val, vc)
    for x in (c, plain, ta, tb, da, db):
        ctx.free(x)
