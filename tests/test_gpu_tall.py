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
