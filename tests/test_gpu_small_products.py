"""Products on either side of the sizes that take fewer launches (1024 tile-rows,
2560 tiles of B, 64 blocks of row classes): C against the oracle, run three times
on one context so that words cleared by a kernel are seen used and cleared again."""
import numpy as np
import pytest

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def matrix(m, n, per_row, seed):
    rng = np.random.default_rng(seed)
    rows = [np.unique(rng.integers(0, n, rng.integers(0, per_row + 1))) for _ in range(m)]
    ptr = np.r_[0, np.cumsum([len(r) for r in rows])]
    return ts.Csr(m, n, ptr, np.concatenate(rows), rng.uniform(-1, 1, ptr[-1]))


@pytest.mark.parametrize("m,k,n,per_row", [(1, 1, 1, 1), (16, 17, 40, 3), (16384, 300, 200, 2), (16385, 300, 200, 2),
                                           (16369, 16384, 16384, 1), (300, 16385, 900, 2), (400, 5000, 3000, 2),
                                           (1000, 16000, 5000, 1), (800, 800, 800, 6), (1024, 1024, 1024, 6), (1025, 1041, 1024, 6)])
@pytest.mark.parametrize("index", [False, True])
def test_small_products(ctx, m, k, n, per_row, index):
    a, b = matrix(m, k, per_row, 1), matrix(k, n, per_row, 2)
    log(f"[small] {m}x{k}x{n} nnz {a.nnz} {b.nnz} index {index}")
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    if index:
        ctx.build_rowindex(ta)
        ctx.build_rowindex(tb)
    rp, cc, vc = oracle.spgemm(a, b)
    for _ in range(3):
        c, st = ctx.spgemm(ta, tb)
        h = ctx.download(ctx.tile2csr(c))
        assert np.array_equal(h.rowptr.astype(np.int64), rp) and np.array_equal(h.colidx, cc) and np.array_equal(h.val, vc)
        assert st.nnzC == rp[-1]
        ctx.free(c)
    for x in (ta, tb, da, db):
        ctx.free(x)
