"""Prefix sums at the edges of their three forms, through tile2csr and
csr2tile of matrices with as many tile-rows, and products whose tile offsets
cross the two- and three-launch sizes."""
import numpy as np
import pytest

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tilem", [1, 15, 16, 16383, 16384, 16385, 20480, 20481])
def test_tile_pointers(ctx, tilem):
    """tile_ptr is a scan of tilem counts: one block up to 16384, two launches above."""
    log(f"[scan] tilem {tilem}")
    m = 16 * tilem - 3
    rng = np.random.default_rng(tilem)
    cnt = rng.integers(0, 3, m)
    ptr = np.concatenate([[0], np.cumsum(cnt)])
    col = np.concatenate([np.arange(c) * 40 + (i % 37) for i, c in enumerate(cnt) if c] + [np.zeros(0, np.int64)])
    a = ts.Csr(m, 150, ptr, col, np.ones(len(col)))
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    got, ref = ctx.download_tiles(t), oracle.csr2tile(a)
    for k in ("tile_ptr", "tile_colidx", "tile_nnz"):
        assert np.array_equal(got[k], ref[k]), k
    ctx.free(t)
    ctx.free(d)


def test_three_launch_scan(ctx):
    """C of a periodic 27-point 144^3 product has 23.3M tiles, more than 4096 blocks of 4096 counts."""
    n = 144
    a = ts.gen_stencil27(n, n, n, True, ts.VAL_KEEP)
    d = ctx.upload(a)
    t = ctx.csr2tile(d)
    ctx.build_csc(t)
    c, st = ctx.spgemm(t, t)
    assert st.nnzC == 125 * n**3 and c.numtile > 4096 * 4096
    o = ctx.tile2csr(c)
    nnz = ctx.host_ints(o.rowptr + 4 * (n**3 - 1), 2)
    assert nnz[1] == st.nnzC and nnz[1] - nnz[0] == 125
    last = ctx.tile_rows_csr(c, [0, n**3 // 2, n**3 - 1])
    assert np.array_equal(np.diff(last.rowptr), [125] * 3)
    for x in (o, c, t, d):
        ctx.free(x)
