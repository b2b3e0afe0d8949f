"""RCM and permutation at the edges of their kernels: 64 and 65 children of
one parent, hubs among levels of short lists, many components, long chains,
rows of 64, 65, 4096 and 4097 entries, one-sided patterns."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def graph(n, edges, seed=0, both=True):
    e = np.asarray(edges, np.int64).reshape(-1, 2)
    r, c = (np.r_[e[:, 0], e[:, 1]], np.r_[e[:, 1], e[:, 0]]) if both else (e[:, 0], e[:, 1])
    p = np.random.default_rng(seed).permutation(n)
    a = sp.coo_matrix((np.ones(len(r)), (p[r], p[c])), shape=(n, n)).tocsr()
    a.data[:] = np.random.default_rng(seed).uniform(-1, 1, a.nnz)
    return ts.Csr.from_scipy(a)


def star(k, at=0):
    return [(at, at + 1 + i) for i in range(k)]


def graphs():
    for k in (63, 64, 65, 200):
        yield f"star{k}", graph(k + 1, star(k))
        # two levels: the hub's children have children of their own
        yield f"tree{k}", graph(1 + k + 3 * k, star(k) + [(1 + i, 1 + k + 3 * i + j) for i in range(k) for j in range(3)])
    yield "chain", graph(700, [(i, i + 1) for i in range(699)])
    yield "chains", graph(3000, [(i, i + 1) for i in range(2999) if i % 7])
    yield "stars", graph(66 * 50, [x for s in range(50) for x in star(40 + s % 26, 66 * s)])
    rng = np.random.default_rng(3)
    yield "one_sided", graph(900, rng.integers(0, 900, (2500, 2)), both=False)
    yield "lower", graph(500, [(i, j) for i in range(500) for j in range(max(0, i - 3), i + 1)], both=False)


@pytest.mark.parametrize("name,a", list(graphs()), ids=[n for n, _ in graphs()])
def test_rcm_edges(ctx, name, a):
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


@pytest.mark.parametrize("longest", [1, 63, 64, 65, 128, 129, 4095, 4096, 4097])
def test_permute_row_lengths(ctx, longest):
    log(f"[permute] longest row {longest}")
    rng = np.random.default_rng(longest)
    n, rows = 4200, 300
    cnt = rng.integers(0, min(longest, 90) + 1, rows)
    cnt[[7, 150, 299]] = longest
    cols = [np.sort(rng.choice(n, c, replace=False)) for c in cnt]
    a = ts.Csr(rows, n, np.r_[0, np.cumsum(cnt)], np.concatenate(cols), rng.uniform(-1, 1, int(cnt.sum())))
    old = rng.permutation(rows).astype(np.int32)
    new = rng.permutation(n).astype(np.int32)
    d = ctx.upload(a)
    p = ctx.permute(d, old, new)
    got = ctx.download(p)
    ref = oracle.permute_csr(a, old, new)
    assert np.array_equal(got.rowptr, ref[0]) and np.array_equal(got.colidx, ref[1]) and np.array_equal(got.val, ref[2])
    ctx.free(p)
    ctx.free(d)
