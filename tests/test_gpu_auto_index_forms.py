"""Products large enough to make their own row indices, of operands that are
not whole tile matrices with every array: without in-tile columns (the drop-in
entry point uploads none), and one operand a part of the other."""
import ctypes as C

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
