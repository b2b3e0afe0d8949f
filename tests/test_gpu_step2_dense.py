"""Step 2 with the window's rows as bits (both block sizes) at the edges of
its rule and windows: spans of 1024 and 4096 tile columns and one more, half
and three fifths of the span filled and just less, empty windows, hub rows,
ragged last tile-rows, views.  Every array of C is compared with the oracle."""
import numpy as np
import pytest

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def csr(m, n, rows):
    ptr = np.zeros(m + 1, np.int64)
    for r, c in rows.items():
        ptr[r + 1] = len(c)
    cols = np.concatenate([np.asarray(rows[r], np.int32) for r in sorted(rows)] + [np.zeros(0, np.int32)])
    return ts.Csr(m, n, np.cumsum(ptr), cols, np.random.default_rng(m).uniform(-1, 1, len(cols)))


def spread(span, tiles, off):
    """One column in each of `tiles` tiles spread over `span` tile columns, first and last included."""
    return np.unique(np.linspace(0, span - 1, tiles).astype(np.int64)) * 16 + off


def inputs():
    rng = np.random.default_rng(11)
    # A: 40 rows over 30 columns of B's rows; B: 30 rows over `span` tile columns
    for span in (1, 63, 1023, 1024, 1025, 4095, 4096, 4097, 9000):
        for fill in (span, (span + 1) // 2, (3 * span + 4) // 5, max(1, span // 2 - 1)):
            b = {r: spread(span, fill, r % 16) for r in range(30)}
            a = {r: np.sort(rng.choice(30, 1 + r % 3, replace=False)) for r in range(39)}
            yield f"span{span}_{fill}", csr(40, 30, a), csr(30, 16 * span, b)
    # windows 1 and 2 of three hold no tile of tile-row 0's C
    yield ("gap", csr(20, 9, {0: [0, 1], 17: [2]}),
           csr(9, 16 * 13000, {0: np.arange(4000) * 16, 1: np.arange(9000, 13000) * 16 + 5, 2: np.arange(13000) * 16}))
    # hub rows of A and of B among short ones; more than 64 entries per wave
    n = 20011
    a = {r: np.sort(rng.choice(n, 3, replace=False)) for r in range(n)}
    a[5] = np.arange(0, n, 3)
    a[8] = np.sort(rng.choice(n, 2500, replace=False))
    a[n - 1] = np.arange(0, n, 7)
    g = csr(n, n, a)
    yield "hub", g, g


@pytest.mark.parametrize("name,a,b", list(inputs()), ids=[i[0] for i in inputs()])
def test_step2_windows(ctx, name, a, b):
    log(f"[step2 dense] {name} A {a.m}x{a.n} nnz {a.nnz} B {b.m}x{b.n} nnz {b.nnz}")
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    plain, _ = ctx.spgemm(ta, tb)  # without row indices: tile pairs
    want = ctx.download_tiles(plain)
    ctx.build_rowindex(ta)
    ctx.build_rowindex(tb)
    c, _ = ctx.spgemm(ta, tb)
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask"):
        assert np.array_equal(got[k], want[k]), k
    assert got["val"].tobytes() == want["val"].tobytes()
    h = ctx.download(ctx.tile2csr(c))
    rp, cc = oracle.spgemm_structure(a, b)
    assert np.array_equal(h.rowptr.astype(np.int64), rp) and np.array_equal(h.colidx, cc)
    if a.m > 16:  # tile-rows 1.. as a view of A
        v, _ = ctx.spgemm_tile_rows(ta, tb, 1, ta.tilem)
        hv = ctx.download(ctx.tile2csr(v))
        assert np.array_equal(hv.rowptr, h.rowptr[16:] - h.rowptr[16])
        assert np.array_equal(hv.colidx, h.colidx[h.rowptr[16]:])
        assert hv.val.tobytes() == h.val[h.rowptr[16]:].tobytes()
        ctx.free(v)
    for x in (c, plain, ta, tb, da, db):
        ctx.free(x)
