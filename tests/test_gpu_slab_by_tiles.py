"""Rows beyond the symbolic table whose C structure is found tile by tile (an A
tile holds five entries or more on average, and an A tile and a B tile carry two
products or more), beside the same rows
found entry by entry: A rows around one chunk of 512 (A tile, B class) slots
and several, C rows past a window of 4096 tile columns, rows of more than 65536
pairs (cut into tasks), light and heavy tiles on either side, empty rows of B,
and B = A^T.  The first call of a handle recomputes the structure, the second
copies the staged lists: both against the oracle."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from

pytestmark = pytest.mark.gpu


def tiled(m, n, h, w, per_row, fill, seed):
    """m x n of h x w tiles: per_row[i] random tiles in tile row i, every entry
    kept with probability `fill`, one at least."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i, p in enumerate(per_row):
        for t in rng.choice(n // w, p, replace=False):
            keep = rng.random(h * w) < fill
            keep[rng.integers(h * w)] = True
            e = np.flatnonzero(keep)
            rows.append(h * i + e // w)
            cols.append(w * t + e % w)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    ok = rows < m
    rows, cols = rows[ok], cols[ok]
    return csr_from(m, n, *(x[np.lexsort((cols, rows))] for x in (rows, cols)),
                    rng.uniform(-1, 1, len(rows)))


def check(gpu, a, b, by_tiles, lb_mode="adaptive-tail", path="vector"):
    pa = gpu.prepare_identity_a(a)
    src = gpu.upload_csr(b)
    ref = oracle.spgemm(as_tuple(a), as_tuple(b))
    pb = gpu.rebuild_b_general(pa, src)
    at, bt = pa.tiles(), pb.tiles()
    fill_a = at["payload_size"] / at["num_tiles"]
    fill_b = bt["payload_size"] / bt["num_tiles"]
    assert (fill_a >= 5.0 and fill_a * fill_b / 4.0 >= 2.0) == by_tiles
    for _ in range(2):
        tc, _ = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path=path, lb_mode=lb_mode))
        check_c(gpu, tc, ref)


@pytest.mark.parametrize("fill_a,fill_b,by_tiles", [(0.9, 0.5, True), (1.0, 0.04, True),
                                                    (0.06, 1.0, False), (0.04, 0.04, False)])
@pytest.mark.parametrize("path", ["vector", "tile"])
def test_chunks_and_windows(gpu, fill_a, fill_b, by_tiles, path):
    a = tiled(30, 1200, 8, 4, [60, 102, 103, 290], fill_a, 1)
    b = tiled(1200, 8 * 6000, 4, 8, np.where(np.arange(300) % 7 == 3, 0, 30), fill_b, 2)
    check(gpu, a, b, by_tiles, path=path)


@pytest.mark.parametrize("lb_mode", ["static", "dynamic", "adaptive-tail"])
def test_rows_cut_into_tasks(gpu, lb_mode):
    per = np.where(np.arange(300) % 10 == 0, 900, 240)
    a = tiled(24, 1200, 8, 4, [290, 30, 250], 0.3, 3)
    check(gpu, a, tiled(1200, 8 * 3000, 4, 8, per, 0.3, 4), True, lb_mode)


@pytest.mark.parametrize("path", ["vector", "auto", "tile"])
def test_transpose(gpu, path):
    """A * A^T with wide rows: B's rows in class order, values in A's payload."""
    n = 8 * 1100
    a = tiled(n, n, 8, 4, np.where(np.arange(1100) % 90 == 5, 700, 4), 0.5, 5)
    pa = gpu.prepare_identity_a(a)
    ref = oracle.spgemm(as_tuple(a), as_tuple(gpu.csr_transpose(a)))
    pb = None
    for _ in range(2):
        pb = gpu.rebuild_b(pa, 1, pb)
        tc, _ = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path=path))
        check_c(gpu, tc, ref)
