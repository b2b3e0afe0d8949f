"""Step 1 with the narrowest bitmap window at its edges (4096 tile columns of B
and one more) and with 1 to 70 kept B tile-rows (eight are loaded together),
beside tile-rows that are not kept: the tile lists of every window width."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [1, 31, 33, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("kept", [1, 7, 8, 9, 64, 65, 70])
def test_windows_agree(ctx, span, kept):
    log(f"[step1 window] {span} tile columns, {kept} kept tile-rows")
    rng = np.random.default_rng(span + kept)
    rows = {}
    for K in range(kept + 5):  # full or half full, then two far columns (never kept)
        t = np.arange(rng.integers(0, 3), span, 1 + K % 2) if K < kept else np.array([0, span - 1])
        rows[16 * K + K % 16] = np.unique(16 * t + K % 16)
    m = 16 * (kept + 5)
    b = ts.Csr(m, 16 * span, np.r_[0, np.cumsum([len(rows.get(r, ())) for r in range(m)])],
               np.concatenate([rows[r] for r in sorted(rows)]), np.ones(sum(map(len, rows.values()))))
    keys = sorted(rows)
    sel = [np.array(keys), np.array(keys[::2]), np.array(keys[-5:]), np.array(keys[:1])]
    a = ts.Csr(49, m, np.r_[0, np.cumsum([len(sel[r // 16]) if r % 16 == 0 else 0 for r in range(49)])], np.concatenate(sel),
               np.ones(sum(map(len, sel))))
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    want = [np.unique(np.concatenate([rows[k] // 16 for k in s])) for s in sel]
    for words in (0, 256, 1024, 2048):
        tune = ts.default_tune()
        tune.s1_window_words = words
        c, _ = ctx.spgemm(ta, tb, tune)
        got = ctx.download_tiles(c)
        assert np.array_equal(got["tile_ptr"], np.r_[0, np.cumsum([len(w) for w in want])]), words
        assert np.array_equal(got["tile_colidx"], np.concatenate(want)), words
        ctx.free(c)
    for x in (ta, tb, da, db):
        ctx.free(x)
