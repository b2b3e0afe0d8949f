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
