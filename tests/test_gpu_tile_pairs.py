"""The tile-pair kernel at the edges of its lists: A rows of 63 to 130 tiles
(groups of 64), C rows past 64 tiles (chunks of 64), rows whose pairs outgrow
the list and the held enumeration, payloads past the LDS stage, and products
small enough to be cut into parts of a row.  Structure bit for bit and values
within the forward bound of the oracle, the same bits on a second call."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from
from test_gpu_tile import split_bound_ok

pytestmark = pytest.mark.gpu


def blocks(m, n, per_row, seed, fill=1.0):
    """Tile rows of 8 rows with per_row[i] tiles of 4 columns each, every
    entry kept with probability `fill`."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i, p in enumerate(per_row):
        for t in np.sort(rng.choice(n // 4, p, replace=False)):
            r, c = np.meshgrid(np.arange(8 * i, min(8 * i + 8, m)), np.arange(4 * t, 4 * t + 4),
                               indexing="ij")
            keep = rng.random(r.shape) < fill
            rows.append(r[keep])
            cols.append(c[keep])
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((cols, rows))
    return csr_from(m, n, rows[order], cols[order], rng.uniform(-1, 1, len(rows)))


CASES = {
    "A rows around 64 tiles": ([63, 64, 65, 1, 127, 128, 129, 130], 640, 3, 400),
    "wide C rows": ([5, 40, 2, 9], 200, 60, 4000),
    "many pairs": ([60] * 5, 260, 40, 320),
    "one row": ([17], 80, 9, 100),
    "sparse tiles": ([30, 70, 3, 11, 50], 320, 12, 700),
    "whole tiles at the A stage's edge": ([11, 12, 13, 2, 4], 60, 8, 90),
}


@pytest.mark.parametrize("precision", ["fp64", "split-bf16"])
@pytest.mark.parametrize("name", list(CASES))
def test_lists(gpu, name, precision):
    per_row, k, per_b, n = CASES[name]
    fill = 0.4 if name == "sparse tiles" else 1.0 if name.startswith("whole") else 0.97
    m = 8 * len(per_row) - 2
    a = blocks(m, k, per_row, 3, fill)
    b = gpu.gen_random(k, n, per_b, 5)
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b_general(pa, gpu.upload_csr(b))
    sched = gpu.schedule(numeric_path="tile", precision=precision)
    tc, st = gpu.tilespgemm(pa, pb, sched)
    ref = oracle.spgemm(as_tuple(a), as_tuple(b))
    if precision == "fp64":
        check_c(gpu, tc, ref)
    else:
        assert split_bound_ok(gpu, a, b, tc, ref)["fwd_max"] <= 1e-12
    # The pairs multiplied: A and B tiles that meet, at a C tile of the row.
    at, bt = pa.tiles(), pb.tiles()
    pairs = 0
    for i in range(tc.tilem):
        cj = set(tc.tile_columnidx[tc.tile_ptr[i]:tc.tile_ptr[i + 1]].tolist())
        for kk in at["tile_col_idx"][at["tile_row_ptr"][i]:at["tile_row_ptr"][i + 1]]:
            js = bt["tile_col_idx"][bt["tile_row_ptr"][kk]:bt["tile_row_ptr"][kk + 1]]
            pairs += sum(1 for j in js.tolist() if j in cj)
    assert st["mfma_pairs"] == pairs
    tc2, _ = gpu.tilespgemm(pa, pb, sched)
    assert np.array_equal(tc.tile_csr_Value.view(np.uint64), tc2.tile_csr_Value.view(np.uint64))


def test_infinities_and_nan_stay_in_their_tiles(gpu):
    """A value that is not finite reaches only entries of C tiles it is
    multiplied into, never the next tile of the list."""
    a = blocks(48, 64, [6] * 6, 11)
    b = gpu.gen_random(64, 90, 30, 12)
    pa = gpu.prepare_identity_a(a)
    src = gpu.upload_csr(b)
    pb = gpu.rebuild_b_general(pa, src)
    sched = gpu.schedule(numeric_path="tile")
    clean, _ = gpu.tilespgemm(pa, pb, sched)
    v = b.val.copy()
    v[7], v[400] = np.inf, np.nan
    src.set_values(v)
    gpu.update_b_values(pa, src, pb)
    tc, _ = gpu.tilespgemm(pa, pb, sched)
    hit = {int(b.col[e]) // 8 for e in (7, 400)}
    tile_of = np.repeat(np.arange(tc.numtile), np.diff(tc.tile_nnz))
    touched = np.isin(tc.tile_columnidx[tile_of], list(hit))
    assert np.array_equal(tc.tile_csr_Value[~touched], clean.tile_csr_Value[~touched])
    assert not np.all(np.isfinite(tc.tile_csr_Value[touched]))
