"""Calls that run out of device memory part of the way: what they took goes
back."""
import pytest

from memory_limit import run_limited

pytestmark = pytest.mark.gpu


def test_tile2csr_gives_back_what_it_took(tmp_path):
    run_limited(tmp_path, """
ctx = ts.Context(0)
a = ts.gen_stencil27(36, 33, 37, valmode=ts.VAL_UNIFORM_PM1, seed=3)
d = ctx.upload(a)
t = ctx.csr2tile(d)
ctx.free(ctx.tile2csr(t))  # the context's scratch exists from here on
ctx.trim()
base, before = limit.limit_live(), ctx.bytes_in_use()
failed = 0
for room in [0, 1 << 10] + [x << 20 for x in (1, 2, 4, 6, 8, 10, 12, 14, 16, 20, 24)]:
    limit.limit_set(base + room)
    for call in (ctx.tile2csr, ctx.build_rowindex):
        if t.rowx_ptr:
            break
        try:
            r = call(t)
            if call == ctx.tile2csr:
                assert np.array_equal(ctx.download(r).val, a.val)
                ctx.free(r)
        except ts.TsgError as e:
            assert e.status == -4, e
            failed += 1
            assert ctx.bytes_in_use() == before, (room, call)
    ctx.trim()
log("failed", failed)
assert failed > 4 and t.rowx_ptr
""")


@pytest.mark.parametrize("matrix", ["ts.gen_stencil27(36, 33, 37, valmode=ts.VAL_UNIFORM_PM1, seed=3)",
                                    "ts.gen_banded(30000, 40, seed=3)"], ids=["mesh", "band"])
@pytest.mark.parametrize("apart", [False, True])
def test_products_index_themselves_only_if_there_is_room(tmp_path, apart, matrix):
    """Wherever the product fits without indices of its own it is computed; what does not fit leaves nothing."""
    run_limited(tmp_path, f"apart, a = {apart}, {matrix}" + """
ctx = ts.Context(0)
d = ctx.upload(a)
ta = ctx.csr2tile(d)
tb = ctx.csr2tile(d) if apart else ta
ctx.build_csc(tb)
plain = ts.default_tune()
plain.element_mode = 1  # no element kernels, so no indices

def product(tune):
    c, _ = ctx.spgemm(ta, tb, tune)
    out = ctx.download_tiles(c)
    ctx.free(c)
    return out

peak = []
for tune in (plain, None):
    for _ in range(2):  # the second time the context's scratch is there
        ctx.trim()
        limit.limit_peak(1)
        want = product(tune)
    peak.append(limit.limit_peak(0))
ctx.trim()
base, before = limit.limit_live(), ctx.bytes_in_use()
log("base", base, "peak without / with indices", peak)
assert peak[1] > peak[0] + 8 * a.nnz
done, refused = [], 0
for room in sorted(set(np.linspace(base, peak[1] + (1 << 20), 24).astype(int)) | {peak[0]}):
    limit.limit_set(int(room))
    ctx.trim()
    try:
        got = product(None)
        for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
            assert np.array_equal(got[k], want[k]), (room, k)
        done.append(room)
    except ts.TsgError as e:
        assert e.status == -4, e
        refused += 1
    assert ctx.bytes_in_use() == before, room
log("done from", min(done), "refused", refused)
assert min(done) <= peak[0] and refused > 0
""")


def test_large_results_without_pinned_memory(tmp_path):
    run_limited(tmp_path, """
ctx = ts.Context(0)
n = 3000001
a = ts.Csr(1, n, np.array([0, n], np.int32), np.arange(n, dtype=np.int32), np.arange(n) * 0.5)
d = ctx.upload(a)
for off in (1, 0, 1):
    limit.limit_no_pinned(off)
    h = ctx.download(d)
    assert np.array_equal(h.rowptr, a.rowptr) and np.array_equal(h.colidx, a.colidx) and np.array_equal(h.val, a.val)
    ctx.trim()
""")


def test_heavy_rows_with_less_room_than_their_windows(tmp_path):
    """The window table of heavy rows (68 MB here) shrinks to what memory there is."""
    run_limited(tmp_path, """
ctx = ts.Context(0)
rng = np.random.default_rng(1)
rows, n = 260, (1 << 26) - 2048  # 65534 windows, one fewer than the most
def csr(m, n, cols):
    ptr = np.r_[0, np.cumsum([len(c) for c in cols])]
    return ts.Csr(m, n, ptr, np.concatenate(cols), rng.uniform(-1, 1, int(ptr[-1])))
b = csr(rows, n, [np.unique(np.r_[0, n - 1, rng.integers(0, n, 40), rng.integers(0, 3000, 60)]) for _ in range(rows)])
a = csr(5, rows, [np.sort(rng.choice(rows, k, replace=False)) for k in (200, 250, 1, 150, 3)])
da, db = ctx.upload(a), ctx.upload(b)
ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
ctx.build_csc(tb)
ctx.build_rowindex(ta)
ctx.build_rowindex(tb)
tune = ts.default_tune()
tune.heavy_min_products = 5000
def product():
    c, st = ctx.spgemm(ta, tb, tune)
    assert st.heavy_rows == 3
    out = ctx.download_tiles(c)
    ctx.free(c)
    return out, st.heavy_bytes
want, table = product()
ctx.trim()
limit.limit_peak(1)
product()
peak = limit.limit_peak(0)
log("peak", peak, "heavy rows' bytes", table)
assert table > 60 << 20
before, least = ctx.bytes_in_use(), table
for less in range(0, int(table * 0.95), 8 << 20):
    ctx.trim()
    limit.limit_set(int(peak - less))
    got, used = product()
    for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "csr_col", "mask", "val"):
        assert np.array_equal(got[k], want[k]), (less, k)
    assert ctx.bytes_in_use() == before
    least = min(least, used)
log("least", least)
assert least < table / 7  # halved three times, plus the rows' lists
""")
