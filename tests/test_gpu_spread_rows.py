"""Numeric rows of products with sparse C tiles (padded accumulator, light
pairs taken row by row) and of products with full ones: rows at the edges of
the accumulator, and every pairing of light and heavy tiles, with B rows of 1
to 8 values whose payload starts inside and past the record."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from, oracle_product

pytestmark = pytest.mark.gpu


def mat(m, n, cells, seed):
    keep = np.unique(np.array([r * n + c for r, c in cells], np.int64))
    rng = np.random.default_rng(seed)
    return csr_from(m, n, keep // n, keep % n, rng.uniform(-1, 1, len(keep)))


def general(gpu, a, b):
    pa = gpu.prepare_identity_a(a)
    src = gpu.upload_csr(b)
    tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b_general(pa, src))
    return tc


@pytest.mark.parametrize("row_nnz", [127, 128, 129, 992, 1023, 1024, 1025])
@pytest.mark.parametrize("step", [1, 3, 8])
def test_accumulator_edges(gpu, row_nnz, step):
    """Tile rows of C with row_nnz entries, `step` columns apart (fill of 8 to
    64 entries a C tile): A is one entry a row, B spreads it."""
    m, n = 64, 8 * 1100
    per = [row_nnz // 8 + (1 if r < row_nnz % 8 else 0) for r in range(8)]
    acells = [(r, r) for r in range(m)]
    bcells = [(r, (c * step + 5 * (r // 8)) % n) for r in range(m) for c in range(per[r % 8])]
    a, b = mat(m, m, acells, 1), mat(m, n, bcells, row_nnz)
    want = oracle.spgemm(as_tuple(a), as_tuple(b))
    check_c(gpu, general(gpu, a, b), want)


@pytest.mark.parametrize("filler", [0, 60])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 5, 8])
def test_light_and_heavy_pairs(gpu, width, filler):
    """B tiles whose rows hold `width` values each, or one row only, against A
    tiles of one column, of two columns and full; `filler` scattered entries a
    row of B keep C's tiles sparse."""
    rng = np.random.default_rng(width * 100 + filler)
    m, k, n = 96, 64, 4096
    acells, bcells = [], []
    for t in range(m // 8):
        for kt in range(k // 4):
            kind = (t + kt) % 5
            cols = {0: [], 1: [kt % 4], 2: [kt % 4], 3: [0, 3], 4: [0, 1, 2, 3]}[kind]
            for c in cols:
                rows = rng.choice(8, {1: 1, 2: 2, 3: 1, 4: 5}[kind], replace=False)
                acells += [(8 * t + int(r), 4 * kt + c) for r in rows]
    for kt in range(k // 4):
        for j in range(6):
            live = [kt % 4] if (kt + j) % 3 == 0 else range(4)
            for kk in live:
                cols = rng.choice(8, width, replace=False) + 8 * (3 * j + kt)
                bcells += [(4 * kt + kk, int(c)) for c in cols]
    for r in range(k):
        bcells += [(r, int(c)) for c in rng.choice(n, filler // 8, replace=False)]
    a, b = mat(m, k, acells, 2), mat(k, n, bcells, 3)
    check_c(gpu, general(gpu, a, b), oracle.spgemm(as_tuple(a), as_tuple(b)))


@pytest.mark.parametrize("g", [3, 9])
def test_stencil_square_and_transpose(gpu, g):
    """27-point boxes, A*A^T (records copied from A's) and A*A."""
    ix = np.arange(g ** 3)
    x, y, z = ix % g, ix // g % g, ix // g ** 2
    cells = []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                ok = ((x + dx >= 0) & (x + dx < g) & (y + dy >= 0) & (y + dy < g) &
                      (z + dz >= 0) & (z + dz < g))
                cells += list(zip(ix[ok], (ix + dx + dy * g + dz * g * g)[ok]))
    a = mat(g ** 3, g ** 3, cells, g)
    pa = gpu.prepare_identity_a(a)
    for aat in (0, 1):
        tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, aat))
        check_c(gpu, tc, oracle_product(a, aat))
