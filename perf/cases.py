"""The work that programs built on this library have it do, as timed cases.

Every case goes through the public Python entry points (rw-spgemm_amd/tilespgemm.py, one ctypes call
per C entry point of include/tsg.h) on matrices that are resident on the GPU.  Kinds:

product   C = A*A or A*A^T on operands already in tile form: what an iterative program repeats
          (Galerkin products, graph powers) and what bench.py times.
operands  CSR -> the operands of a product: tiles, the CSC tile index, the element row index and,
          for A*A^T, the transpose.  Paid once per new matrix.
csr       C's tiles -> CSR, what a program does to hand C on.
whole     CSR in, CSR out: operands, product, CSR of C, everything else released.
reorder   RCM order of a matrix and P*A*P^T, the reorder path before a product.
batch     many small products in one captured graph, then every C fetched as a host CSR.

Matrix families: 5-point and 27-point grids (periodic and Dirichlet; banded tiles, few entries each),
Erdos-Renyi (hypersparse tiles), banded (dense tiles) and R-MAT (hub rows).  Values are float64, the
library's only value type.
"""
import math
import os
import sys
import zlib

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rw-spgemm_amd"))
import tilespgemm as ts  # noqa: E402

DEV = "cuda:0"
_ctx = None


def context():
    """One context for the process, as a program holds it (a stream and a caching allocator)."""
    global _ctx
    if _ctx is None:
        _ctx = ts.Context(0)
    return _ctx


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest call: the 64x64 Laplacian of the library's smoke test; launches and latency
        {"name": "product_a2_5pt_64", "kind": "product", "op": "a2", "family": "grid5", "nx": 64, "ny": 64},
        # the headline: periodic 27-point 128^3 (bench.py)
        {"name": "product_a2_27p_128", "kind": "product", "op": "a2", "family": "grid27", "nx": 128, "ny": 128, "nz": 128, "periodic": True},
        # an ordinary mesh with odd sides: tile boundaries fall anywhere in a grid line
        {"name": "product_a2_27d_61x47x53", "kind": "product", "op": "a2", "family": "grid27", "nx": 61, "ny": 47, "nz": 53, "periodic": False},
        # the largest random problems of the batched workload: hypersparse tiles
        {"name": "product_a2_er_65521", "kind": "product", "op": "a2", "family": "er", "n": 65521, "mean": 18.0},
        # the batched workload's banded problems: tiles nearly full
        {"name": "product_aat_band_39989", "kind": "product", "op": "aat", "family": "band", "n": 39989, "half": 20},
        # a power-law graph: hub rows carry most of the products
        {"name": "product_aat_rmat_16", "kind": "product", "op": "aat", "family": "rmat", "scale": 16, "ef": 16},
        # a new mesh matrix arrives: its operands for A^2
        {"name": "operands_a2_27p_96", "kind": "operands", "op": "a2", "family": "grid27", "nx": 96, "ny": 96, "nz": 96, "periodic": True},
        # a new graph arrives (the served workload's larger matrices): its operands for A*A^T
        {"name": "operands_aat_rmat_18", "kind": "operands", "op": "aat", "family": "rmat", "scale": 18, "ef": 16},
        # C of a mesh product handed on as CSR
        {"name": "csr_27d_79x83x81", "kind": "csr", "op": "a2", "family": "grid27", "nx": 79, "ny": 83, "nz": 81, "periodic": False},
        # one product on a new random matrix, CSR to CSR
        {"name": "whole_aat_er_20011", "kind": "whole", "op": "aat", "family": "er", "n": 20011, "mean": 12.0},
        # a mesh whose rows arrive in no useful order: RCM and permutation
        {"name": "reorder_27d_61x64x59", "kind": "reorder", "op": "a2", "family": "grid27", "nx": 61, "ny": 64, "nz": 59, "periodic": False, "shuffled": True},
        # many small products per step: half random, half banded, half A^2, half A*A^T
        {"name": "batch_20", "kind": "batch", "count": 20, "nmin": 1000, "nmax": 8191},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["product", "product", "product", "product", "operands", "operands", "csr", "whole", "whole", "reorder", "batch"])
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 20), "nmin": _log(rng, 200, 1500), "nmax": _log(rng, 2000, 8000)}
    family = rng.choice(["grid27", "er", "band", "rmat"] + (["grid5"] if kind != "reorder" else []))
    c = {"kind": kind, "op": rng.choice(["a2", "aat"]), "family": family}
    # rows: a product's C and a whole call's are many times the operand
    top = {"product": 1.0, "operands": 2.0, "csr": 0.5, "whole": 0.5, "reorder": 0.12}[kind]
    if family == "grid5":
        c |= {"nx": _log(rng, 64, 1200), "ny": _log(rng, 64, max(80, int(800 * top)))}
    elif family == "grid27":
        hi = 110 * top ** (1.0 / 3)
        c |= {"nx": _log(rng, 12, hi), "ny": _log(rng, 12, hi), "nz": _log(rng, 12, hi), "periodic": rng.random() < 0.5}
    elif family == "er":
        c |= {"n": _log(rng, 1000, 65536 * top), "mean": round(rng.uniform(4, 26), 1)}
    elif family == "band":
        c |= {"n": _log(rng, 1000, 100000 * top), "half": rng.randint(2, 40)}
    else:
        c |= {"scale": rng.randint(11, {"product": 16, "operands": 18, "csr": 14, "whole": 15, "reorder": 14}[kind]), "ef": rng.randint(6, 16)}
    if kind == "reorder":
        c["shuffled"] = True
        if family == "band":  # its levels are n / half: a chain of dependent launches
            c["half"] = rng.randint(20, 40)
    return c


# ------------------------------------------------------------------ inputs, made on the GPU
def _csr_of_keys(keys, n):
    """rowptr, colidx of the sorted distinct keys row * n + column."""
    row = torch.div(keys, n, rounding_mode="floor")
    col = (keys - row * n).to(torch.int32)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return ptr.to(torch.int32), col


def _grid_keys(case):
    dims = [case["nx"], case["ny"]] + ([case["nz"]] if case["family"] == "grid27" else [])
    n = math.prod(dims)
    at = torch.arange(n, dtype=torch.int64, device=DEV)
    coord, rest = [], at
    for d in dims:
        coord.append(rest % d)
        rest = torch.div(rest, d, rounding_mode="floor")
    if case["family"] == "grid5":
        offs = [(0, 0), (-1, 0), (1, 0), (0, -1), (0, 1)]
    else:
        offs = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
    cols = torch.empty(n, len(offs), dtype=torch.int64, device=DEV)
    for j, o in enumerate(offs):
        ok = torch.ones(n, dtype=torch.bool, device=DEV)
        col, stride = torch.zeros(n, dtype=torch.int64, device=DEV), 1
        for d, x, k in zip(dims, coord, o):
            y = x + k
            if case.get("periodic"):
                y = y % d
            else:
                ok &= (y >= 0) & (y < d)
            col += y * stride
            stride *= d
        cols[:, j] = torch.where(ok, at * n + col, n * n)
    cols = torch.sort(cols, 1)[0].reshape(-1)
    cols = cols[cols < n * n]
    keep = torch.ones_like(cols, dtype=torch.bool)
    keep[1:] = cols[1:] != cols[:-1]
    return cols[keep], n


def _moved(keys, n, to):
    """Rows and columns i of the keys renumbered to[i]."""
    row = torch.div(keys, n, rounding_mode="floor")
    return torch.sort(to[row] * n + to[keys - row * n])[0]


def make_csr(case, seed):
    """n, rowptr, colidx (int32) and val (float64) of the case's square matrix, on the GPU.

    A random pattern is drawn for the case's sizes and its blocks of 16 rows and columns are then
    renumbered by the seed: other seeds give other matrices with as many entries and tiles in A and C.
    """
    g = torch.Generator(device=DEV)
    g.manual_seed(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k not in ("name", "kind", "op"))).encode()))
    h = torch.Generator(device=DEV)
    h.manual_seed(int(seed))
    family = case["family"]
    if family in ("grid5", "grid27"):
        keys, n = _grid_keys(case)
    elif family == "er":
        n = case["n"]
        cnt = torch.poisson(torch.full((n,), float(case["mean"]), device=DEV), generator=g).to(torch.int64)
        row = torch.repeat_interleave(torch.arange(n, device=DEV), cnt)
        keys = torch.unique(row * n + torch.randint(0, n, row.shape, generator=g, device=DEV))
        at = torch.arange(n, device=DEV)
        whole = n // 16  # a last, shorter block stays where it is
        block = torch.randperm(whole, generator=h, device=DEV)
        at[:16 * whole] = (16 * block[:, None] + torch.arange(16, device=DEV)[None, :]).reshape(-1)
        keys = _moved(keys, n, at)
    elif family == "band":
        n, w = case["n"], 2 * case["half"] + 1
        col = torch.arange(n, device=DEV)[:, None] + torch.arange(w, device=DEV)[None, :] - case["half"]
        row = torch.arange(n, device=DEV)[:, None].expand(n, w)
        keys = (row * n + col)[(col >= 0) & (col < n)]
    else:
        n = 1 << case["scale"]
        u = torch.zeros(n * case["ef"], dtype=torch.int64, device=DEV)
        v = torch.zeros_like(u)
        for _ in range(case["scale"]):  # quadrants 0.57, 0.19, 0.19, 0.05
            p = torch.rand(u.shape, generator=g, device=DEV)
            u = 2 * u + (p >= 0.76).long()
            v = 2 * v + (((p >= 0.57) & (p < 0.76)) | (p >= 0.95)).long()
        keys = torch.unique(torch.cat([u * n + v, v * n + u]))
        flip = int(torch.randint(0, n // 16, (1,), generator=h, device=DEV)) * 16  # keeps the quadrants' nesting
        keys = _moved(keys, n, torch.arange(n, device=DEV) ^ flip)
    if case.get("shuffled"):
        keys = _moved(keys, n, torch.randperm(n, generator=h, device=DEV))
    ptr, col = _csr_of_keys(keys, n)
    val = torch.rand(col.shape, generator=h, device=DEV, dtype=torch.float64)
    val = 1.0 - val if family == "rmat" else 2.0 * val - 1.0
    return n, ptr, col, val


def _dcsr(n, ptr, col, val):
    return ts.DCsr(n, n, int(col.numel()), ptr.data_ptr(), col.data_ptr(), val.data_ptr())


# ------------------------------------------------------------------ what the library hands back
class _Device:
    def __init__(self, p, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (p or 0, False), "version": 2}


def _view(p, n, typestr):
    return torch.as_tensor(_Device(p, n, typestr), device=DEV)


def _tiles_out(t):
    nt = t.numtile
    return {"tile_ptr": _view(t.tile_ptr, t.tilem + 1, "<i4"), "tile_colidx": _view(t.tile_colidx, nt, "<i4"),
            "tile_nnz": _view(t.tile_nnz, nt + 1, "<i4"), "csr_ptr": _view(t.csr_ptr, 16 * nt, "|u1"),
            "csr_col": _view(t.csr_col, t.nnz, "|u1"), "val": _view(t.val, t.nnz, "<f8"),
            "mask": _view(t.mask, 16 * nt, "<i2")}


def _operand_out(t):
    out = _tiles_out(t)
    if t.csc_ptr:
        out |= {"csc_ptr": _view(t.csc_ptr, t.tilen + 1, "<i4"), "csc_rowidx": _view(t.csc_rowidx, t.numtile, "<i4"),
                "csc_tileid": _view(t.csc_tileid, t.numtile, "<i4")}
    if t.rowx_ptr:
        out |= {"rowx_ptr": _view(t.rowx_ptr, t.m + 1, "<i4"), "rowx_col": _view(t.rowx_col, t.nnz, "<i4"),
                "rowx_val": _view(t.rowx_val, t.nnz, "<f8")}
    return out


def _csr_out(d):
    return {"rowptr": _view(d.rowptr, d.m + 1, "<i4"), "colidx": _view(d.colidx, d.nnz, "<i4"),
            "val": _view(d.val, d.nnz, "<f8")}


# ------------------------------------------------------------------ states
class State:
    """The inputs and device objects of one case; what a pass returns stays until the next pass."""

    def __init__(self, case):
        self.case = case
        self.owned = []   # library objects kept for the state's life
        self.last = []    # the previous pass's results
        self.batch = None

    def drop_last(self):
        ctx = context()
        for o in self.last:
            ctx.free(o)
        self.last = []

    def __del__(self):
        if _ctx is None:
            return
        if self.batch is not None:
            self.batch.close()
        for o in self.last + self.owned:
            _ctx.free(o)


def operands(ctx, a, op):
    """(tiles of A, tiles of B) with every index a product uses; B is A itself for A^2."""
    ta = ctx.csr2tile(a)
    if op == "a2":
        ctx.build_csc(ta)
        ctx.build_rowindex(ta)
        return ta, ta
    at = ctx.transpose(a)
    tb = ctx.csr2tile(at)
    ctx.build_csc(tb)
    ctx.build_rowindex(tb)
    ctx.build_rowindex(ta)
    ctx.free(at)
    return ta, tb


def _batch_problem(case, i):
    """Problem i's matrix case and operation: sizes spread evenly over log n, fixed by the case alone."""
    f = i / max(1, case["count"] - 1)
    n = int(round(case["nmin"] * (case["nmax"] / case["nmin"]) ** f)) | 1
    if i % 2:
        return {"family": "er", "n": n, "mean": float(4 + (5 * i) % 24)}, "a2" if i % 4 == 1 else "aat"
    return {"family": "band", "n": n, "half": 2 + (7 * i) % 38}, "a2" if i % 4 == 0 else "aat"


def prepare(case, seed):
    ctx = context()
    s = State(case)
    if case["kind"] == "batch":
        made = [make_csr(_batch_problem(case, i)[0], seed * 1000 + i) for i in range(case["count"])]
        torch.cuda.synchronize()
        ops = [ts.OP_A2 if _batch_problem(case, i)[1] == "a2" else ts.OP_AAT for i in range(case["count"])]
        s.batch = ts.Batch(ctx, [_dcsr(*m) for m in made], ops)
        return s
    s.keep = make_csr(case, seed)
    torch.cuda.synchronize()
    s.a = _dcsr(*s.keep)
    if case["kind"] in ("product", "csr"):
        s.ta, s.tb = operands(ctx, s.a, case["op"])
        s.owned = [s.ta] if s.tb is s.ta else [s.ta, s.tb]
        s.keep = s.a = None  # the tiles are all that the program goes on with
        if case["kind"] == "csr":
            s.tc, _ = ctx.spgemm(s.ta, s.tb, timed=False)
            s.owned.append(s.tc)
        ctx.sync()
    return s


def run(s):
    ctx, kind = context(), s.case["kind"]
    if kind == "batch":
        s.batch.run()
        out = {}
        for i in range(s.case["count"]):
            c = s.batch.result_csr(i)
            out["%02d" % i] = {"rowptr": c.rowptr, "colidx": c.colidx, "val": c.val}
        return out
    s.drop_last()
    if kind == "product":
        c, _ = ctx.spgemm(s.ta, s.tb, timed=False)
        s.last = [c]
        return _tiles_out(c)
    if kind == "operands":
        ta, tb = operands(ctx, s.a, s.case["op"])
        s.last = [ta] if tb is ta else [ta, tb]
        return [_operand_out(t) for t in s.last]
    if kind == "csr":
        c = ctx.tile2csr(s.tc)
        s.last = [c]
        return _csr_out(c)
    if kind == "whole":
        ta, tb = operands(ctx, s.a, s.case["op"])
        tc, _ = ctx.spgemm(ta, tb, timed=False)
        c = ctx.tile2csr(tc)
        ctx.free(tc)
        if tb is not ta:
            ctx.free(tb)
        ctx.free(ta)
        s.last = [c]
        return _csr_out(c)
    old, levels = ctx.order_rcm(s.a)
    new = np.empty_like(old)
    new[old] = np.arange(old.size, dtype=old.dtype)
    p = ctx.permute(s.a, old, new)
    s.last = [p]
    return {"order": old, "levels": levels, **_csr_out(p)}


# ------------------------------------------------------------------ what a pass cannot do without
def _tile_bytes(n, tiles, nnz):
    return 4 * (n // 16 + 2) + 8 * tiles + 48 * tiles + 9 * nnz


def _er_tiles(n, per_row):
    """Expected 16x16 tiles hit by n * per_row uniform entries."""
    nt = (n / 16.0) ** 2
    return nt * -math.expm1(-n * per_row / nt)


def _shape(case):
    """Rows, entries and tiles of A; products, entries and tiles of C (expected values for random matrices)."""
    f = case["family"]
    if f == "grid5":
        n = case["nx"] * case["ny"]
        return n, 5 * n, n // 16 * 5, 25 * n, 13 * n, n // 16 * 10
    if f == "grid27":
        n = case["nx"] * case["ny"] * case["nz"]
        e = [1.0 if case["periodic"] else 1 - 2 / (3.0 * case[k]) for k in ("nx", "ny", "nz")]
        e2 = [1.0 if case["periodic"] else 1 - 6 / (5.0 * case[k]) for k in ("nx", "ny", "nz")]
        one, two = math.prod(e), math.prod(e2)
        return n, 27 * n * one, n / 16 * 27 * one, 729 * n * one * one, 125 * n * two, n / 16 * 125 * two
    if f == "er":
        n, d = case["n"], case["mean"]
        c = n * -math.expm1(-d * d / n)
        return n, n * d, _er_tiles(n, d), n * d * d, n * c, _er_tiles(n, c)
    if f == "band":
        n, h = case["n"], case["half"]
        return n, n * (2 * h + 1), n / 16 * (h / 8 + 2), n * (2 * h + 1.0) ** 2, n * (4 * h + 1), n / 16 * (h / 4 + 2)
    n, e = 1 << case["scale"], case["ef"] / 16.0  # fitted to generated R-MAT graphs
    nnz = 1.85 * case["ef"] * n * (0.95 + 0.008 * (case["scale"] - 18))
    prod = 9.5e9 * (e * e) * 2.72 ** (case["scale"] - 18)
    nnzc = min(prod, 2.9e9 * e * 2.75 ** (case["scale"] - 18))
    return n, nnz, 0.6 * nnz, prod, nnzc, nnzc / 8


def work(case):
    if case["kind"] == "batch":
        b = fl = 0.0
        for i in range(case["count"]):
            n, nnz, t, prod, nnzc, tc = _shape(_batch_problem(case, i)[0])
            b += _tile_bytes(n, t, nnz) + 4 * n + 12 * nnzc
            fl += 2 * prod
        return {"bytes": b, "flops": fl}
    n, nnz, t, prod, nnzc, tc = _shape(case)
    twice = 2 if case["op"] == "aat" else 1
    csr_a, csr_c = 4 * n + 12 * nnz, 4 * n + 12 * nnzc
    if case["kind"] == "product":
        return {"bytes": twice * _tile_bytes(n, t, nnz) + _tile_bytes(n, tc, nnzc), "flops": 2 * prod}
    if case["kind"] == "operands":
        return {"bytes": csr_a + twice * (_tile_bytes(n, t, nnz) + csr_a) + 8 * t, "flops": 0}
    if case["kind"] == "csr":
        return {"bytes": _tile_bytes(n, tc, nnzc) - 32 * tc + csr_c, "flops": 0}
    if case["kind"] == "whole":
        return {"bytes": csr_a + csr_c, "flops": 2 * prod}
    return {"bytes": 2 * csr_a + 4 * n, "flops": 0}


# ------------------------------------------------------------------ the same results in plain torch
def _transpose(n, ptr, col, val):
    row = torch.repeat_interleave(torch.arange(n, device=DEV), (ptr[1:] - ptr[:-1]).long())
    order = torch.argsort(col.long() * n + row)
    cnt = torch.bincount(col.long(), minlength=n)
    tp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    tp[1:] = torch.cumsum(cnt, 0)
    return tp, row[order], val[order]


def _tile_key(row, col, n):
    tn = (n + 15) // 16
    return (((row // 16) * tn + col // 16) * 16 + row % 16) * 16 + col % 16


def _product_values(case, seed, tiled):
    """C's values, in tile order or in CSR order: products of a few rows at a time, summed in 64 bits."""
    n, ptr, col, val = make_csr(case, seed)
    ptr, col = ptr.long(), col.long()
    bp, bc, bv = (ptr, col, val) if case["op"] == "a2" else _transpose(n, ptr, col, val)
    blen = bp[1:] - bp[:-1]
    per = torch.zeros(col.numel() + 1, dtype=torch.int64, device=DEV)
    per[1:] = torch.cumsum(blen[col], 0)
    by_row = per[ptr].cpu().numpy()
    host_ptr = ptr.cpu().numpy()
    out, r0 = [], 0
    while r0 < n:
        r1 = int(np.searchsorted(by_row, by_row[r0] + (1 << 26), side="right")) - 1
        r1 = min(n, max(r0 + 16, r1 // 16 * 16))
        e0, e1 = int(host_ptr[r0]), int(host_ptr[r1])
        k, a = col[e0:e1], val[e0:e1]
        row = torch.repeat_interleave(torch.arange(r0, r1, device=DEV), ptr[r0 + 1:r1 + 1] - ptr[r0:r1])
        ln = blen[k]
        tot = int(ln.sum())
        if tot:
            src = torch.repeat_interleave(torch.arange(e1 - e0, device=DEV), ln)
            first = torch.cumsum(ln, 0) - ln
            e = torch.arange(tot, device=DEV) - first[src] + bp[k][src]
            rr, cc = row[src], bc[e]
            key = _tile_key(rr, cc, n) if tiled else rr * n + cc
            key, inv = torch.unique(key, return_inverse=True)
            out.append(torch.zeros(key.numel(), dtype=torch.float64, device=DEV).index_add_(0, inv, a[src] * bv[e]))
        r0 = r1
    return torch.cat(out) if out else torch.zeros(0, dtype=torch.float64, device=DEV)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return {"%02d" % i: {"rowptr": None, "colidx": None, "val": _product_values(dict(p, op=op), seed * 1000 + i, False)}
                for i in range(case["count"]) for p, op in [_batch_problem(case, i)]}
    if kind == "product":
        return {"val": _product_values(case, seed, True)}
    if kind in ("csr", "whole"):
        return {"val": _product_values(case, seed, False)}
    n, ptr, col, val = make_csr(case, seed)
    row = torch.repeat_interleave(torch.arange(n, device=DEV), (ptr[1:] - ptr[:-1]).long())
    if kind == "operands":
        tiles = {"val": val[torch.argsort(_tile_key(row, col.long(), n))], "rowx_val": val}
        if case["op"] == "a2":
            return [tiles]
        tp, tc, tv = _transpose(n, ptr, col, val)
        trow = torch.repeat_interleave(torch.arange(n, device=DEV), tp[1:] - tp[:-1])
        return [tiles, {"val": tv[torch.argsort(_tile_key(trow, tc, n))], "rowx_val": tv}]
    return None  # reorder: the order is whole numbers, the values are moved
