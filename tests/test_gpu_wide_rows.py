"""Tile-pair rows of many C tiles, which take their pairs a few C tiles at a
time: rows around the limit (64 C tiles) beside narrow ones, A rows of one and
several groups of 64 tiles, dense rows (a list of two C tiles) and sparse ones
with B tiles between C's columns that meet nothing, rows cut into units, light
and heavy tiles, B = A^T, heavy tiles left to the tail queue, split precision
and the allocation-free call.  Structure bit for bit and values within the
forward bound of the oracle, every pair once, the same bits on a second call."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c
from test_gpu_slab_by_tiles import tiled
from test_gpu_tile import split_bound_ok
from test_zz_no_alloc import values_into_buffer

pytestmark = pytest.mark.gpu


def pairs_met(pa, pb, tc):
    """A and B tiles that meet, at a C tile of the row."""
    at, bt = pa.tiles(), pb.tiles()
    n = 0
    for i in range(tc.tilem):
        cj = tc.tile_columnidx[tc.tile_ptr[i]:tc.tile_ptr[i + 1]]
        for k in at["tile_col_idx"][at["tile_row_ptr"][i]:at["tile_row_ptr"][i + 1]]:
            js = bt["tile_col_idx"][bt["tile_row_ptr"][k]:bt["tile_row_ptr"][k + 1]]
            n += int(np.isin(js, cj).sum())
    return n


def check(gpu, a, b, precision="fp64", **kw):
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b_general(pa, gpu.upload_csr(b))
    sched = gpu.schedule(numeric_path="tile", precision=precision, **kw)
    tc, st = gpu.tilespgemm(pa, pb, sched)
    ref = oracle.spgemm(as_tuple(a), as_tuple(b))
    if precision == "fp64":
        check_c(gpu, tc, ref)
    else:
        assert split_bound_ok(gpu, a, b, tc, ref)["fwd_max"] <= 1e-12
    again, _ = gpu.tilespgemm(pa, pb, sched)
    assert np.array_equal(tc.tile_csr_Value.view(np.uint64), again.tile_csr_Value.view(np.uint64))
    return pa, pb, tc, st


#         A tiles per row, B rows (4 each), B tiles per row, C tile columns, fills
CASES = {
    "around the limit": ([1, 2, 3, 5, 1, 0, 4], 8, 33, 90, 0.9, 0.9),
    "groups of A tiles": ([63, 64, 65, 130, 1, 191], 200, 40, 400, 0.6, 0.6),
    "dense": ([128, 70, 129], 130, 130, 130, 1.0, 1.0),
    "few meet": ([70, 140, 9], 220, 60, 900, 0.04, 0.04),
    "light A, full B": ([70, 30, 200], 220, 50, 700, 0.03, 1.0),
    "units": ([90], 100, 700, 2000, 0.5, 0.3),
}


@pytest.mark.parametrize("precision", ["fp64", "split-bf16"])
@pytest.mark.parametrize("name", list(CASES))
def test_wide_rows(gpu, name, precision):
    per_a, kt, per_b, nt, fill_a, fill_b = CASES[name]
    a = tiled(8 * len(per_a) - 3, 4 * kt, 8, 4, per_a, fill_a, 1)
    rng = np.random.default_rng(2)
    rows = np.minimum(nt, rng.integers(max(1, per_b // 2), per_b + 1, kt))
    if name == "dense":
        rows[:] = nt
    b = tiled(4 * kt, 8 * nt - 5, 4, 8, np.minimum(rows, nt - 1), fill_b, 3)
    pa, pb, tc, st = check(gpu, a, b, precision)
    assert st["mfma_pairs"] == pairs_met(pa, pb, tc)
    assert np.diff(tc.tile_ptr).max() > 64
    # The allocation-free call takes the same units.
    got = values_into_buffer(gpu, pa, pb, precision, tc.nnz)
    assert np.array_equal(got.view(np.uint64), tc.tile_csr_Value.view(np.uint64))


@pytest.mark.parametrize("precision", ["fp64", "split-bf16"])
def test_heavy_tiles_are_left_to_the_tail_queue(gpu, precision):
    a = tiled(24, 4 * 300, 8, 4, [200, 150, 20], 0.7, 5)
    b = tiled(4 * 300, 8 * 200, 4, 8, np.full(300, 60), 0.7, 6)
    plain = check(gpu, a, b, precision)[2]
    _, _, tc, st = check(gpu, a, b, precision, split_threshold=330.0, split_chunk_target=100.0,
                         force_tail_split=1)
    assert st["tail_reason"] == 1 and 0 < st["tail_records"] < tc.numtile
    assert np.array_equal(tc.tile_columnidx, plain.tile_columnidx)


@pytest.mark.parametrize("fill", [0.0, 12.0])
def test_transpose_and_mixed_rows(gpu, fill):
    """A * A^T, and rows of the other kernels beside wide ones."""
    n = 8 * 300
    per = np.where(np.arange(300) % 23 == 4, 200, 3)
    a = tiled(n, n, 8, 4, per, 0.6, 7)
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b(pa, 1)
    ref = oracle.spgemm(as_tuple(a), as_tuple(gpu.csr_transpose(a)))
    tc, _ = gpu.tilespgemm(pa, pb, gpu.schedule(tile_fill_threshold=fill))
    check_c(gpu, tc, ref)
