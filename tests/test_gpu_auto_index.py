"""Products of operands without row indices, large enough that the product
makes its own: the same C as on the tile-pair path, the operands and the
context's memory as before, with either operand indexed, both, one matrix as
both operands in one struct and in two, and A and B apart."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu

KEYS = ("tile_ptr", "tile_colidx", "tile_rowidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val")


@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("index_a,index_b", [(False, False), (True, False), (False, True), (True, True)])
def test_products_index_themselves(ctx, apart, index_a, index_b):
    a = ts.gen_stencil27(36, 33, 37, valmode=ts.VAL_UNIFORM_PM1, seed=3)
    log(f"[auto index] nnz {a.nnz} apart {apart} index {index_a} {index_b}")
    assert a.nnz >= 1 << 20
    b = ts.Csr(a.m, a.n, a.rowptr, a.colidx, np.random.default_rng(2).uniform(-1, 1, a.nnz)) if apart else a
    da, db = ctx.upload(a), ctx.upload(b)
    ta = ctx.csr2tile(da)
    tb = ctx.csr2tile(db) if apart or index_a != index_b else ta
    ctx.build_csc(tb)
    if index_a:
        ctx.build_rowindex(ta)
    if index_b:
        ctx.build_rowindex(tb)
    tune = ts.default_tune()
    tune.force_tile_parallel = 1
    plain, _ = ctx.spgemm(ta, tb, tune)
    want = ctx.download_tiles(plain)
    before = bool(ta.rowx_ptr), bool(tb.rowx_ptr), ctx.bytes_in_use()
    for _ in range(2):
        c, _ = ctx.spgemm(ta, tb)
        got = ctx.download_tiles(c)
        for k in KEYS:
            assert np.array_equal(got[k], want[k]), k
        ctx.free(c)
        assert (bool(ta.rowx_ptr), bool(tb.rowx_ptr), ctx.bytes_in_use()) == before
    for x in (plain, ta, da, db) + ((tb,) if tb is not ta else ()):
        ctx.free(x)
