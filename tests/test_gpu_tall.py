"""Matrices with so many rows that 16, 64 or 256 threads a row are more than the
2^32 of a launch: nearly all rows empty, results known from the rest."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def rowptr_of(m, rows, counts):
    """Row pointers of m rows, `counts` entries in the ascending rows `rows`."""
    p = np.zeros(m + 1, np.int32)
    p[rows + 1] = counts
    np.cumsum(p, out=p)
    return p


@pytest.mark.parametrize("m,longest", [((1 << 24) + 5, 70), ((1 << 24) + 5, 4096), ((1 << 26) + 3, 9)])
def test_permute(ctx, m, longest):
    """Up to 64 entries one wave a row, up to 4096 one block."""
    log(f"[tall] permute {m} rows, longest {longest}")
    rng = np.random.default_rng(longest)
    n = 5000
    rows = np.unique(np.r_[0, 3, m // 2, m - 2, m - 1, rng.integers(0, m, 200)])
    counts = rng.integers(1, min(longest, 60) + 1, len(rows)).astype(np.int32)
    counts[[0, len(rows) // 2, -1]] = longest
    cols = np.concatenate([np.sort(rng.choice(n, c, replace=False)) for c in counts])
    a = ts.Csr(m, n, rowptr_of(m, rows, counts), cols, rng.uniform(-1, 1, len(cols)))
    old = np.roll(np.arange(m, dtype=np.int32), 12345)  # row r of the result is row r - 12345
    new = rng.permutation(n).astype(np.int32)
    d = ctx.upload(a)
    p = ctx.permute(d, old, new)
    got = ctx.download(p)
    ctx.free(p)
    ctx.free(d)
    at = (rows.astype(np.int64) + 12345) % m
    order = np.argsort(at)
    small = ts.Csr(len(rows), n, np.r_[0, np.cumsum(counts)], cols, a.val)
    ref = oracle.permute_csr(small, order.astype(np.int32), new)
    assert np.array_equal(got.rowptr, rowptr_of(m, at[order], counts[order]))
    assert np.array_equal(got.colidx, ref[1]) and np.array_equal(got.val, ref[2])


def test_rcm_and_permute(ctx):
    """2^28 vertices, nearly all isolated; a clique whose first vertex has more than 64 children, a star of
    more than 4096, a path."""
    n = (1 << 28) + 7
    rng = np.random.default_rng(5)
    k = 70 + 4200 + 300
    ids = np.sort(np.unique(np.r_[1, n - 1, rng.integers(0, n, 2 * k)])[:k])
    ids[-1] = n - 1
    v = rng.permutation(k)
    edges = [(v[i], v[j]) for i in range(70) for j in range(i)]
    edges += [(v[70], v[71 + i]) for i in range(4199)]
    edges += [(v[4270 + i], v[4271 + i]) for i in range(299)]
    e = np.asarray(edges)
    s = sp.coo_matrix((np.ones(2 * len(e)), (np.r_[e[:, 0], e[:, 1]], np.r_[e[:, 1], e[:, 0]])), shape=(k, k)).tocsr()
    s.data[:] = rng.uniform(-1, 1, s.nnz)
    small = ts.Csr.from_scipy(s)
    a = ts.Csr(n, n, rowptr_of(n, ids, np.diff(small.rowptr)), ids[small.colidx], small.val)
    log(f"[tall] rcm {n} vertices, {a.nnz} entries")
    d = ctx.upload(a)
    order, _ = ctx.order_rcm(d)
    want = oracle.rcm(small)
    assert np.array_equal(order[:k], ids[want])
    alone = np.ones(n, bool)  # the others: isolated, by descending id
    alone[ids] = False
    assert np.array_equal(order[k:], np.flatnonzero(alone)[::-1])
    log("[tall] order checked")
    new = np.empty(n, np.int32)
    new[order] = np.arange(n, dtype=np.int32)
    p = ctx.permute(d, order, new)
    got = ctx.download(p)
    ctx.free(p)
    ctx.free(d)
    ctx.trim()
    inv = np.empty(k, np.int32)
    inv[want] = np.arange(k, dtype=np.int32)
    ref = oracle.permute_csr(small, want.astype(np.int32), inv)
    assert np.array_equal(got.rowptr[:k + 1], ref[0]) and np.all(got.rowptr[k:] == a.nnz)
    assert np.array_equal(got.colidx, ref[1]) and np.array_equal(got.val, ref[2])


@pytest.mark.parametrize("log_rows", [23, 24])
@pytest.mark.parametrize("mode,heavy", [(0, 0), (0, 2000), (2, 0), (None, 0)])
def test_product(ctx, log_rows, mode, heavy):
    """2^23 and 2^24 tile-rows, of which some dozens have entries: some for row lines, some element-wise, some
    with heavy rows; mode None without A's row index.  C is the C of those tile-rows alone."""
    rng = np.random.default_rng(11)
    n, tilem = 4000, (1 << log_rows) + 5
    m = 16 * tilem - 3
    b = ts.gen_er(n, 20.0, seed=4)
    at = np.unique(np.r_[0, 1, tilem // 2, tilem - 1, rng.integers(0, tilem, 40)])  # tile-rows with entries
    counts = rng.integers(0, 4, 16 * len(at)).astype(np.int32)
    counts[16 * 3:16 * 6] = 40  # their C rows are long
    counts[16 * 9 + 2] = 600
    counts[-3:] = 0  # past the last row
    cols = np.concatenate([np.sort(rng.choice(n, c, replace=False)) for c in counts])
    val = rng.uniform(-1, 1, len(cols))
    rows = (16 * at[:, None] + np.arange(16)[None, :]).ravel()
    tall = ts.Csr(m, n, rowptr_of(m, rows[:-3], counts[:-3]), cols, val)
    small = ts.Csr(16 * len(at), n, np.r_[0, np.cumsum(counts)], cols, val)
    log(f"[tall] product, {tilem} tile-rows, mode {mode}, heavy from {heavy}")
    db = ctx.upload(b)
    tb = ctx.csr2tile(db)
    ctx.build_csc(tb)
    ctx.build_rowindex(tb)
    tune = ts.default_tune()
    tune.element_mode = mode or 0
    tune.heavy_min_products = heavy
    out = []
    for a in (tall, small):  # in this order: C of the first is not left where the second's goes
        da = ctx.upload(a)
        ta = ctx.csr2tile(da)
        if mode is not None:
            ctx.build_rowindex(ta)
        c, st = ctx.spgemm(ta, tb, tune)
        out.append((ctx.download_tiles(c), st.heavy_rows))
        for x in (c, ta, da):
            ctx.free(x)
    ctx.free(tb)
    ctx.free(db)
    ctx.trim()
    (got, hg), (want, hw) = out
    assert hw == hg and (heavy == 0 or hg > 0)
    ptr = np.zeros(tilem + 1, np.int32)
    ptr[at + 1] = np.diff(want["tile_ptr"])
    assert np.array_equal(got["tile_ptr"], np.cumsum(ptr))
    assert np.array_equal(got["tile_rowidx"], at[want["tile_rowidx"]])
    for k in ("tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
        assert np.array_equal(got[k], want[k]), k
