"""Conversions at the edges of their work split: runs of 1024 tiles of a
tile-row, batches of 64 tiles or 448 entries, full tiles, ragged last
tile-rows, tile-row views.  Every array is compared with the oracle, bit for
bit."""
import numpy as np
import pytest

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def csr(m, n, rows):
    """CSR of {row: sorted columns}; distinct values."""
    ptr = np.zeros(m + 1, np.int64)
    for r, c in rows.items():
        ptr[r + 1] = len(c)
    cols = np.concatenate([np.asarray(rows[r], np.int32) for r in sorted(rows)] + [np.zeros(0, np.int32)])
    return ts.Csr(m, n, np.cumsum(ptr), cols, np.arange(1, len(cols) + 1, dtype=np.float64) / 3)


def inputs():
    rng = np.random.default_rng(5)

    def some(n, k):
        return np.sort(rng.choice(n, k, replace=False))

    # one tile-row of exactly t tiles (one entry each), rows above and below it
    for t in (64, 65, 1024, 1025, 2049):
        yield f"tiles{t}", csr(50, 16 * t + 5, {3: [7], 20: np.arange(t) * 16 + 3, 21: [0, 16 * t - 1], 49: [1, 2]})
    # a hub row among short ones: more than 4096 entries in its tile-row, in several runs of tiles
    yield "hub", csr(37, 40001, {**{r: some(40001, 40) for r in range(37)}, 5: np.arange(0, 40001, 2), 33: np.arange(40001)})
    # full tiles: 448 entries are one tile and three quarters; ragged sides
    yield "dense70", csr(70, 75, {r: np.arange(75) for r in range(70)})
    # tiles of 224 entries: two fill a batch exactly; and of 225
    for k in (14, 15):
        yield f"fill{k}", csr(16, 160, {r: np.concatenate([np.arange(16 * j, 16 * j + k) for j in range(10)]) for r in range(16)})
    # wide rows: bitmap windows of 8192 tile columns
    yield "wide", csr(18, 600011, {r: some(600011, 3 + 50 * (r % 3)) for r in range(18)})
    yield "wide_hub", csr(18, 600011, {2: some(600011, 9000), 3: some(600011, 5), 17: [600010]})
    # columns near the end of the int32 range
    top = 2**31 - 32
    yield "int32_columns", csr(3, top, {0: [0, top - 40, top - 1], 1: [5, top - 2], 2: [top - 17, top - 16, top - 1]})
    yield "one", csr(1, 1, {0: [0]})
    yield "norows", csr(0, 5, {})


@pytest.mark.parametrize("name,a", list(inputs()), ids=[n for n, _ in inputs()])
def test_conversion_edges(ctx, name, a):
    log(f"[convert] {name} {a.m}x{a.n} nnz {a.nnz}")
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    got = ctx.download_tiles(t)
    ref = oracle.csr2tile(a, packed=False)
    for k in ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "val", "mask"):
        assert np.array_equal(got[k], ref[k]), k
    back = ctx.tile2csr(t)
    h = ctx.download(back)
    assert np.array_equal(h.rowptr, a.rowptr) and np.array_equal(h.colidx, a.colidx) and np.array_equal(h.val, a.val)
    for o in (back, t, d):
        ctx.free(o)


@pytest.mark.parametrize("name,a", list(inputs()), ids=[n for n, _ in inputs()])
def test_transpose_and_csc_edges(ctx, name, a):
    """The stable transpose and the CSC tile index of the same matrices (row starts across blocks of 4096 entries)."""
    if name == "int32_columns":
        pytest.skip("a transpose of 2^31 rows is not of interest")
    log(f"[transpose] {name}")
    d = ctx.upload(a)
    dt = ctx.transpose(d)
    t = ctx.download(dt)
    tp, tc, tv = oracle.transpose(a)
    assert np.array_equal(t.rowptr, tp) and np.array_equal(t.colidx, tc) and np.array_equal(t.val, tv)
    tt = ctx.transpose(dt)
    b = ctx.download(tt)
    assert np.array_equal(b.rowptr, a.rowptr) and np.array_equal(b.colidx, a.colidx) and np.array_equal(b.val, a.val)
    ta = ctx.csr2tile(d)
    ctx.build_csc(ta)
    got = ctx.download_tiles(ta)
    order = np.lexsort((got["tile_rowidx"], got["tile_colidx"]))
    assert np.array_equal(got["csc_tileid"], order) and np.array_equal(got["csc_rowidx"], got["tile_rowidx"][order])
    assert np.array_equal(got["csc_ptr"], np.concatenate([[0], np.cumsum(np.bincount(got["tile_colidx"], minlength=ta.tilen))]))
    for o in (ta, tt, dt, d):
        ctx.free(o)


def test_transpose_with_long_runs_of_empty_rows(ctx):
    """More rows start in a block of entries than are marked: rows found by search."""
    a = csr(50001, 3000, {0: [5, 9], 1: np.arange(2000), 40000: [1], 40001: np.arange(0, 3000, 2), 50000: np.arange(700)})
    d = ctx.upload(a)
    dt = ctx.transpose(d)
    t = ctx.download(dt)
    tp, tc, tv = oracle.transpose(a)
    assert np.array_equal(t.rowptr, tp) and np.array_equal(t.colidx, tc) and np.array_equal(t.val, tv)
    ctx.free(dt)
    ctx.free(d)


def test_tile2csr_of_a_view(ctx):
    """Tile-rows [1, 3) of a matrix as a view: its own rows, whatever tile count the view carries."""
    a = csr(60, 40000, {**{r: np.arange(r, 40000, 97) for r in range(60)}, 18: np.arange(0, 40000, 3)})
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    v = ts.DTiles.from_buffer_copy(t)
    v.tile_ptr = t.tile_ptr + 4
    v.m, v.tilem = 32, 2
    for numtile in (t.numtile, 1):
        v.numtile = numtile
        o = ctx.tile2csr(v)
        h = ctx.download(o)
        ctx.free(o)
        lo, hi = a.rowptr[16], a.rowptr[48]
        assert np.array_equal(h.rowptr, a.rowptr[16:49] - lo)
        assert np.array_equal(h.colidx, a.colidx[lo:hi]) and np.array_equal(h.val, a.val[lo:hi])
    ctx.free(t)
    ctx.free(d)


def test_tile2csr_ignores_offsets_past_the_rows(ctx):
    """Row offsets of the last tile-row past the matrix's rows are not read (a caller's own tiles may hold anything)."""
    a = csr(21, 90, {r: np.arange(r % 5, 90, 1 + r % 4) for r in range(21)})
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    h = ctx.download_tiles(t)
    p = h["csr_ptr"].reshape(-1, 16).copy()
    p[h["tile_ptr"][1]:, 5:] = 0
    raw = np.ascontiguousarray(p).reshape(-1)
    assert ts.lib.tsg_h2d(ctx.h, t.csr_ptr, raw.ctypes.data, raw.size) == 0
    o = ctx.tile2csr(t)
    b = ctx.download(o)
    assert np.array_equal(b.rowptr, a.rowptr) and np.array_equal(b.colidx, a.colidx) and np.array_equal(b.val, a.val)
    for x in (o, t, d):
        ctx.free(x)


def test_check_accepts_row_starts_anywhere(ctx):
    """Descending columns across row starts at every place of a block of 4096 entries; long runs of empty rows."""
    n = 5000
    rows = {0: np.arange(4095), 1: np.arange(4096), 2: [0], 3: [n - 1], 4: [0], 5: np.arange(3000), 20009: np.arange(1095), 20010: [7]}
    a = csr(40011, n, rows)
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    o = ctx.tile2csr(t)
    b = ctx.download(o)
    assert np.array_equal(b.rowptr, a.rowptr) and np.array_equal(b.colidx, a.colidx) and np.array_equal(b.val, a.val)
    for x in (o, t, d):
        ctx.free(x)


@pytest.mark.parametrize("what", ["descending", "repeated", "column", "negative", "rowptr", "total", "hub"])
def test_bad_csr_is_refused(ctx, what):
    """Unsorted, repeated and out-of-range columns and inconsistent row pointers stay errors."""
    a = csr(40, 9000, {**{r: np.arange(r, 9000, 311) for r in range(40)}, 7: np.arange(9000)})
    rp, ci = a.rowptr.copy(), a.colidx.copy()
    if what == "descending":
        ci[[5, 6]] = ci[[6, 5]]
    elif what == "repeated":
        ci[6] = ci[5]
    elif what == "column":
        ci[rp[40] - 1] = 9000
    elif what == "negative":
        ci[rp[21]] = -1
    elif what == "rowptr":
        rp[16], rp[17] = rp[17], rp[16]
    elif what == "total":
        rp[40] -= 1
    else:
        ci[rp[7] + 5000] = ci[rp[7] + 4999]
    d = ctx.upload(ts.Csr(40, 9000, rp, ci, a.val))
    d.nnz = a.nnz
    for call in (ctx.csr2tile, ctx.transpose):
        with pytest.raises(ts.TsgError) as e:
            call(d)
        assert e.value.status == -2
    ctx.free(d)
