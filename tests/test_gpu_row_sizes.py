"""C's sizes and the numeric routing at the edges of their pass: tile-row
counts around its 1024-row workgroups and the look-back's 64-workgroup step,
rows that go through every symbolic pass in one call, handles that size C
again after a smaller and a larger product, and thresholds that move rows
between the kernels of one handle."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from

pytestmark = pytest.mark.gpu


def band(n, width, seed):
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(n), width)
    cols = np.clip(rows + np.tile(np.arange(width) - width // 2, n), 0, n - 1)
    keep = np.unique(rows.astype(np.int64) * n + cols)
    return csr_from(n, n, keep // n, keep % n, rng.uniform(-1, 1, len(keep)))


@pytest.mark.parametrize("tile_rows", [1, 255, 1023, 1024, 1025, 64 * 1024, 64 * 1024 + 1, 130 * 1024 + 3])
def test_tile_row_counts(gpu, tile_rows):
    a = band(8 * tile_rows - 3, 3, tile_rows)
    pa = gpu.prepare_identity_a(a)
    tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0))
    check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(a)))


def test_every_symbolic_pass_and_a_handle_reused(gpu):
    """Rows of the wave table, of the workgroup table and of the slab in one
    product, then other B operands on the same A handle."""
    rng = np.random.default_rng(2)
    m, k, n = 700, 600, 60000
    per = np.where(np.arange(m) % 50 == 7, 120, np.where(np.arange(m) % 9 == 0, 30, 2))
    rows = np.repeat(np.arange(m), per)
    cols = np.concatenate([np.sort(rng.choice(k, p, replace=False)) for p in per])
    a = csr_from(m, k, rows, cols, rng.uniform(-1, 1, len(rows)))
    pa = gpu.prepare_identity_a(a)
    for per_b in (40, 1, 60, 3):
        b = gpu.gen_random(k, n, per_b, per_b)
        tc, st = gpu.tilespgemm(pa, gpu.rebuild_b_general(pa, gpu.upload_csr(b)))
        check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(b)))
    big = gpu.gen_random(k, n, 60, 60)
    _, st = gpu.tilespgemm(pa, gpu.rebuild_b_general(pa, gpu.upload_csr(big)))
    assert st["heavy_rows"] > 0


def test_thresholds_on_one_handle(gpu):
    """Every fill threshold routes by its own count, in any order of calls."""
    a = gpu.gen_banded(900, 12, 14, 3)
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b(pa, 0)
    ref = oracle.spgemm(as_tuple(a), as_tuple(a))
    seen = []
    for fill in (12.0, 1.0, 32.0, 12.0, 9.0):
        tc, st = gpu.tilespgemm(pa, pb, gpu.schedule(tile_fill_threshold=fill))
        check_c(gpu, tc, ref)
        seen.append(st["numeric_path"])
    assert seen[1] == gpu.NUMERIC_PATHS["tile"] and seen[2] == gpu.NUMERIC_PATHS["vector"]
    assert seen[0] == seen[3]
