"""Step 2 of tile-rows with many A tiles on either side of the rule that takes
them element-wise (128 tiles, 64 entries a tile), for spans of one small, one
large and several windows.  Every array of C against the tile-pair path."""
import numpy as np
import pytest

import tilespgemm as ts
from tsg_check import log

pytestmark = pytest.mark.gpu


def inputs():
    for tiles in (128, 129):
        for ents in (5, 64, 65):
            for span in (300, 1500, 5000):
                yield tiles, ents, span


@pytest.mark.parametrize("tiles,ents,span", list(inputs()))
def test_many_a_tiles(ctx, tiles, ents, span):
    log(f"[step2 many] {tiles} A tiles of {ents} entries, {span} tile columns")
    rng = np.random.default_rng(tiles + ents)
    # A: one tile-row, `ents` entries in each of its tiles
    keys = np.concatenate([np.sort(rng.choice(256, ents, replace=False)) + 256 * t for t in range(tiles)])
    row, col = keys % 256 // 16, keys // 256 * 16 + keys % 16
    order = np.lexsort((col, row))
    a = ts.Csr(16, 16 * tiles, np.r_[0, np.cumsum(np.bincount(row, minlength=16))], col[order], rng.uniform(-1, 1, len(col)))
    # B: at most 512 C tiles in 300, filled spans otherwise
    cols = [np.sort(rng.choice(16 * span, 40, replace=False)) for _ in range(16 * tiles)]
    b = ts.Csr(16 * tiles, 16 * span, np.arange(0, 40 * 16 * tiles + 1, 40), np.concatenate(cols), rng.uniform(-1, 1, 640 * tiles))
    da, db = ctx.upload(a), ctx.upload(b)
    ta, tb = ctx.csr2tile(da), ctx.csr2tile(db)
    ctx.build_csc(tb)
    tune = ts.default_tune()
    tune.force_tile_parallel = 1
    plain, _ = ctx.spgemm(ta, tb, tune)
    want = ctx.download_tiles(plain)
    ctx.build_rowindex(ta)
    ctx.build_rowindex(tb)
    c, _ = ctx.spgemm(ta, tb)
    got = ctx.download_tiles(c)
    for k in ("tile_ptr", "tile_colidx", "tile_nnz", "csr_ptr", "mask", "csr_col", "val"):
        assert np.array_equal(got[k], want[k]), k
    for x in (c, plain, ta, tb, da, db):
        ctx.free(x)
