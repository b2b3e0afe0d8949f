"""Products large enough to make their own row indices, of operands that are
not whole tile matrices with every array: without in-tile columns (the drop-in
entry point uploads none), and one operand a part of the other."""
import ctypes as C
import time

import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu

KEYS = ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val")


def mesh(seed=3):
    a = ts.gen_stencil27(36, 33, 37, valmode=ts.VAL_UNIFORM_PM1, seed=seed)
    assert a.nnz >= 1 << 20
    return a


def tile_parallel(ctx, ta, tb):
    tune = ts.default_tune()
    tune.force_tile_parallel = 1
    c, _ = ctx.spgemm(ta, tb, tune)
    out = ctx.download_tiles(c)
    ctx.free(c)
    return out


def same_tiles(got, want):
    for k in KEYS:
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("bare_a,bare_b", [(True, False), (False, True), (True, True)])
def test_operands_without_in_tile_columns(ctx, bare_a, bare_b):
    a = mesh()
    log(f"[auto index] no csr_col: A {bare_a} B {bare_b}")
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    ctx.build_csc(t)
    want = tile_parallel(ctx, t, t)
    held = []

    def bare():
        """t again through the CSC tile order, which carries no columns when its input has none"""
        o = ctx.csc_order(t)
        given = ts.DTiles.from_buffer_copy(o)
        given.csr_col = None
        r = ctx.from_csc_order(given)
        held.extend([o, r])
        assert not r.csr_col
        return r

    ta, tb = bare() if bare_a else t, bare() if bare_b else t
    for _ in range(2):
        c, _ = ctx.spgemm(ta, tb)
        same_tiles(ctx.download_tiles(c), want)
        ctx.free(c)
    for x in held + [t, d]:
        ctx.free(x)


@pytest.mark.parametrize("csr_a,csr_b", [(False, True), (True, False), (False, False)])
def test_drop_in_operands_without_csr(csr_a, csr_b):
    """The drop-in entry point on matrices whose CSR arrays are gone once their tiles are made."""
    a = mesh()
    log(f"[auto index] drop-in, CSR kept: A {csr_a} B {csr_b}")
    a.val[:] = np.arange(a.nnz) % 10 + 1
    pair = [ts.HostSMatrix(a), ts.HostSMatrix(a)]
    A, B = pair[0].s, pair[1].s
    ts.lib.csr2tile_row_major(C.byref(A))
    ts.lib.csr2tile_col_major(C.byref(B))
    for s, kept in ((A, csr_a), (B, csr_b)):
        if not kept:
            s.rowpointer = s.columnindex = None
            s.value = None
    Cm = ts.SMatrix()
    out = [C.c_ulonglong()] + [C.c_double() for _ in range(7)]
    ts.lib.tilespgemm(C.byref(A), C.byref(B), C.byref(Cm), None, None, 0, 0.0, 0.0, 1, *[C.byref(x) for x in out[:4]],
                      b"test", *[C.byref(x) for x in out[4:]])
    ts.lib.tile2csr(C.byref(Cm))
    got = [np.ctypeslib.as_array(p, shape=(n,)) for p, n in ((Cm.rowpointer, a.m + 1), (Cm.columnindex, Cm.nnz), (Cm.value, Cm.nnz))]
    want = a.to_scipy() @ a.to_scipy()  # whole numbers: exact
    want.sort_indices()
    assert np.array_equal(got[0], want.indptr) and np.array_equal(got[1], want.indices) and np.array_equal(got[2], want.data)
    ts.lib.matrix_destroy(C.byref(A))
    ts.lib.matrix_destroy(C.byref(B))
    ts.lib.matrix_destroy(C.byref(Cm))
    libc = C.CDLL(None)
    libc.free.argtypes = [C.c_void_p]
    for p in (Cm.rowpointer, Cm.columnindex, Cm.value):
        libc.free(C.cast(p, C.c_void_p))


@pytest.mark.parametrize("index_a,index_b", [(False, False), (True, False), (False, True)])
def test_leading_tile_rows_of_b(ctx, index_a, index_b):
    """A = B's first tile-rows: B's arrays with smaller sizes."""
    a = mesh()
    d = ctx.upload(a)
    tb = ctx.csr2tile(d)
    ctx.build_csc(tb)
    host = ctx.download_tiles(tb)
    want = tile_parallel(ctx, tb, tb)
    ta = ts.DTiles.from_buffer_copy(tb)
    ta.tilem = 2700
    ta.m = 16 * ta.tilem
    ta.numtile = int(host["tile_ptr"][ta.tilem])
    ta.nnz = int(host["tile_nnz"][ta.numtile])
    assert ta.m < tb.m and ta.nnz >= 1 << 20
    log(f"[auto index] {ta.tilem} of {tb.tilem} tile-rows, index {index_a} {index_b}")
    ta.csc_ptr = ta.csc_rowidx = ta.csc_tileid = None
    if index_a:
        ctx.build_rowindex(ta)
    if index_b:
        ctx.build_rowindex(tb)
    nt = int(want["tile_ptr"][ta.tilem])
    nz = int(want["tile_nnz"][nt])
    cut = {"tile_ptr": ta.tilem + 1, "tile_colidx": nt, "tile_rowidx": nt, "tile_nnz": nt + 1, "csr_ptr": 16 * nt,
           "csr_col": nz, "mask": 16 * nt, "val": nz}
    for _ in range(2):
        c, _ = ctx.spgemm(ta, tb)
        got = ctx.download_tiles(c)
        for k in KEYS:
            assert np.array_equal(got[k], want[k][:cut[k]]), k
        ctx.free(c)
    if index_a:
        for p in (ta.rowx_ptr, ta.rowx_col, ta.rowx_val):
            ctx.dfree(p)
    ctx.free(tb)
    ctx.free(d)


def test_operands_that_share_values_only(ctx):
    """B = A one tile column to the right: every array A's but the tile columns."""
    a = mesh()
    d = ctx.upload(a)
    ta = ctx.csr2tile(d)
    ctx.build_csc(ta)
    host = ctx.download_tiles(ta)
    tb = ts.DTiles.from_buffer_copy(ta)
    tb.n, tb.tilen = ta.n + 16, ta.tilen + 1
    tb.csc_ptr = tb.csc_rowidx = tb.csc_tileid = None
    tb.tile_colidx = ctx.dev_ints(host["tile_colidx"] + 1)
    ctx.build_csc(tb)
    want = tile_parallel(ctx, ta, tb)
    c, _ = ctx.spgemm(ta, tb)
    same_tiles(ctx.download_tiles(c), want)
    ctx.free(c)
    for p in (tb.tile_colidx, tb.csc_ptr, tb.csc_rowidx, tb.csc_tileid):
        ctx.dfree(p)
    ctx.free(ta)
    ctx.free(d)


def bands(n, widths, ends):
    """Rows up to ends[i] hold every column within widths[i]."""
    half = np.zeros(n, np.int64)
    for w, lo, hi in zip(widths, [0] + ends[:-1], ends):
        half[lo:hi] = w
    i = np.arange(n)
    first, last = np.maximum(i - half, 0), np.minimum(i + half, n - 1)
    ptr = np.r_[0, np.cumsum(np.maximum(last - first + 1, 0))]
    col = np.arange(ptr[-1]) - np.repeat(ptr[:-1], np.diff(ptr)) + np.repeat(first, np.diff(ptr))
    return ts.Csr(n, n, ptr, col, np.random.default_rng(n).uniform(-1, 1, len(col)))


def dense_tiles(tile_rows, tiles, entries, seed=0):
    """`tiles` tiles of `entries` entries in each tile-row, anywhere."""
    rng = np.random.default_rng(seed)
    n = 16 * tile_rows
    key = np.unique(np.repeat(np.arange(tile_rows), tiles) * tile_rows + rng.integers(0, tile_rows, tile_rows * tiles))
    at = np.argsort(rng.random((len(key), 256)), axis=1)[:, :entries]
    key = np.sort(((key[:, None] // tile_rows * 16 + at // 16) * n + key[:, None] % tile_rows * 16 + at % 16).ravel())
    return ts.Csr(n, n, np.r_[0, np.cumsum(np.bincount(key // n, minlength=n))], key % n, rng.uniform(-1, 1, len(key)))


DENSE = {
    "all_by_lines": lambda: bands(30000, [40], [30000]),
    "few_not": lambda: bands(30000, [20, 100, 20], [10000, 10300, 30000]),  # those as segments
    "one_in_ten_not": lambda: bands(200000, [5, 70, 5], [50000, 70000, 200000]),  # those by tiles, beside the lines
    "half_not": lambda: bands(30000, [10, 64], [15000, 30000]),
    "none": lambda: dense_tiles(3000, 8, 48),
    "none_long_lists": lambda: dense_tiles(1500, 24, 32),
    "some_empty_rows": lambda: bands(60000, [40, -1, 6], [20000, 40000, 60000]),
}


@pytest.mark.parametrize("index_a,index_b", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("name", list(DENSE))
def test_dense_tiles(ctx, name, index_a, index_b):
    """Tiles that meet in dozens of products: the index is made after step 2, or not, by what goes by row lines."""
    a = DENSE[name]()
    assert a.nnz >= 1 << 20 and a.nnz <= 96 * a.m
    log(f"[auto index] dense, {name}: nnz {a.nnz} index {index_a} {index_b}")
    b = ts.Csr(a.m, a.n, a.rowptr, a.colidx, np.random.default_rng(2).uniform(-1, 1, a.nnz))
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    want = tile_parallel(ctx, ta, tb)
    if index_a:
        ctx.build_rowindex(ta)
    if index_b:
        ctx.build_rowindex(tb)
    before = ctx.bytes_in_use()
    for _ in range(2):
        c, _ = ctx.spgemm(ta, tb)
        same_tiles(ctx.download_tiles(c), want)
        ctx.free(c)
        assert ctx.bytes_in_use() == before
    for x in (ta, tb, da, db):
        ctx.free(x)


def best_ms(ctx, t, tune):
    best = 1e9
    for _ in range(8):
        ctx.sync()
        t0 = time.perf_counter()
        c, _ = ctx.spgemm(t, t, tune, timed=False)
        ctx.sync()
        best = min(best, time.perf_counter() - t0)
        ctx.free(c)
    return best * 1e3


@pytest.mark.parametrize("name,least", [("none", 1.5), ("half_not", 1.5)])
def test_index_is_no_loss_on_dense_tiles(ctx, name, least):
    """Against the product that may make none: element by element the first took 1.8 times as long."""
    d = ctx.upload(DENSE[name]())
    t = ctx.csr2tile(d)
    ctx.build_csc(t)
    without = ts.default_tune()
    without.element_mode = 1
    w, m = best_ms(ctx, t, without), best_ms(ctx, t, None)
    log(f"[auto index] {name}: {m:.3f} ms, without an index {w:.3f}")
    assert m <= least * w
    ctx.free(t)
    ctx.free(d)
