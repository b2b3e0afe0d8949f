"""Arrays handed over by the library: small ones are copies, large ones the
library's own memory, freed once and only after the last array on it."""
import gc

import numpy as np
import pytest

import tilespgemm as ts


@pytest.mark.parametrize("nx", [8, 200, 520])  # 520^2 rows: rowptr, colidx and val are all above 1 MiB
def test_arrays_outlive_the_matrix(nx):
    a = ts.gen_stencil5(nx, nx)
    want = (a.rowptr.copy(), a.colidx.copy(), a.val.copy())
    tail, col, ptr = a.val[a.nnz // 2:], a.colidx, a.rowptr
    del a
    gc.collect()
    for _ in range(3):  # the same sizes again, over whatever was freed
        b = ts.gen_stencil5(nx, nx)
        b.val[:] = 0.0
        b.colidx[:] = 0
        del b
    assert np.array_equal(ptr, want[0]) and np.array_equal(col, want[1])
    assert np.array_equal(tail, want[2][len(want[2]) - len(tail):])
    assert ptr.flags.writeable and col.flags.c_contiguous and tail.dtype == np.float64


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 262143, 262144, 262145, 524288, 2097152, 2097153, 9437189])
def test_large_copies_to_the_host(ctx, n):
    """One row of n entries: below and at one piece (2 MiB), more pieces than slots, a ragged last piece."""
    a = ts.Csr(1, n, np.array([0, n], np.int32), np.arange(n, dtype=np.int32), np.arange(n) * 0.5)
    d = ctx.upload(a)
    for _ in range(2):
        h = ctx.download(d)
        assert np.array_equal(h.rowptr, a.rowptr) and np.array_equal(h.colidx, a.colidx) and np.array_equal(h.val, a.val)
    ctx.free(d)
