"""RCM of large sparse graphs whose lists are all short (few lanes a vertex):
many components, chains, lists of the longest length that still counts as
short and one more, vertices alone; permutation of matrices with 16 entries a
row or fewer on average; against the oracle."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def graph(n, edges, both=True, diag=None, seed=0):
    e = np.asarray(edges, np.int64).reshape(-1, 2)
    r, c = (np.r_[e[:, 0], e[:, 1]], np.r_[e[:, 1], e[:, 0]]) if both else (e[:, 0], e[:, 1])
    if diag is not None:
        r, c = np.r_[r, diag], np.r_[c, diag]
    p = np.random.default_rng(seed).permutation(n)
    a = sp.coo_matrix((np.ones(len(r)), (p[r], p[c])), shape=(n, n)).tocsr()
    a.data[:] = np.random.default_rng(seed).uniform(-1, 1, a.nnz)
    return ts.Csr.from_scipy(a)


def stars(n, k):
    """Stars of k leaves, as many as fit."""
    hub = np.arange(n // (k + 1)) * (k + 1)
    return np.c_[np.repeat(hub, k), (hub[:, None] + 1 + np.arange(k)[None, :]).ravel()]


def chains(n, k):
    i = np.arange(n - 1)
    i = i[i % k != k - 1]
    return np.c_[i, i + 1]


N = (1 << 18) + 37  # from 2^18 rows on the union is done by few lanes too
GRAPHS = {
    "alone": lambda: graph(N, [], diag=np.arange(0, N, 3)),
    "pairs": lambda: graph(N, chains(N, 2)),
    "chains9": lambda: graph(N, chains(N, 9), diag=np.arange(N)),
    "one_sided": lambda: graph(N, np.random.default_rng(1).integers(0, N, (N, 2)), both=False),
    "stars31": lambda: graph(N, stars(N, 31)),
    "stars63": lambda: graph(N, stars(N, 63)),
    "stars64": lambda: graph(N, stars(N, 64)),
    "stars65": lambda: graph(N, stars(N, 65)),
    "one_star32": lambda: graph(N, np.r_[chains(N - 40, 5), N - 40 + stars(40, 32)]),
    "one_star33": lambda: graph(N, np.r_[chains(N - 40, 5), N - 40 + stars(40, 33)]),
    "small": lambda: graph(5000, chains(5000, 4), diag=np.arange(0, 5000, 7)),
    "grid": lambda: ts.gen_stencil5(90, 70),
    "tiny": lambda: graph(3, [(0, 1)]),
}


@pytest.mark.parametrize("name", list(GRAPHS))
def test_rcm_short_lists(ctx, name):
    a = GRAPHS[name]()
    log(f"[rcm] {name} n {a.m} nnz {a.nnz}")
    d = ctx.upload(a)
    g = ctx.symmetrize(d)
    h = ctx.download(g)
    gp, gc = oracle.symmetrize(a)
    assert np.array_equal(h.rowptr, gp) and np.array_equal(h.colidx, gc)
    order, _ = ctx.order_rcm(d)
    assert np.array_equal(order, oracle.rcm(a))
    ctx.free(g)
    ctx.free(d)


@pytest.mark.parametrize("longest,some", [(0, 0), (1, 1), (15, 3), (16, 9), (17, 9), (32, 40), (33, 40), (48, 7), (49, 7), (63, 5),
                                          (64, 200), (65, 1), (65, 200), (4096, 3), (4097, 2)])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 700])
def test_permute_short_rows(ctx, rows, longest, some):
    """`some` rows of `longest` entries among rows of 0 to 6, a last row of any length among them."""
    rng = np.random.default_rng(longest * 1000 + rows)
    n = 4500
    cnt = rng.integers(0, 7, rows)
    cnt[rng.choice(rows, min(some, rows), replace=False)] = longest
    cols = [np.sort(rng.choice(n, c, replace=False)) for c in cnt]
    if longest:
        for c in cols[-1:]:
            c[-1:] = n - 1
    a = ts.Csr(rows, n, np.r_[0, np.cumsum(cnt)], np.concatenate(cols), rng.uniform(-1, 1, int(cnt.sum())))
    log(f"[permute] {rows} rows, nnz {a.nnz}, longest {cnt.max()}")
    old, new = rng.permutation(rows).astype(np.int32), rng.permutation(n).astype(np.int32)
    d = ctx.upload(a)
    before = ctx.bytes_in_use()
    p = ctx.permute(d, old, new)
    got = ctx.download(p)
    ref = oracle.permute_csr(a, old, new)
    assert np.array_equal(got.rowptr, ref[0]) and np.array_equal(got.colidx, ref[1]) and np.array_equal(got.val, ref[2])
    ctx.free(p)
    assert ctx.bytes_in_use() == before
    ctx.free(d)
