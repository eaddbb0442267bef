"""Products with a few rows beyond the LDS tables: only those rows and the rows
of B that they select are laid out entry by entry, against the oracle at both
sides of the rule (a sixteenth of A's tile rows and of its slots), for B = A, B = A^T in column
order and in class order, an independent B and a reordered A; with hub rows
that select every row, rows past the numeric tables only, dense and empty
tiles; and the memory that one such row may take."""
import ctypes

import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from

pytestmark = pytest.mark.gpu


def with_wide_rows(n, per, wide, per_wide, seed, block=False):
    """n x n, `per` entries a row, per_wide more in the rows `wide`; block: a
    stretch of full tiles in them too."""
    rng = np.random.default_rng(seed)
    rows = [np.repeat(np.arange(n), per)]
    cols = [rng.integers(0, n, n * per)]
    for i in wide:
        c = rng.choice(n, min(n, per_wide), replace=False)
        if block:
            c = np.r_[c, np.arange(200, 260)]
        rows.append(np.full(len(c), i))
        cols.append(c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    key = np.unique(rows.astype(np.int64) * n + cols)
    rows, cols = key // n, key % n
    return csr_from(n, n, rows, cols, rng.uniform(-1, 1, len(rows)))


N = 8 * 1500   # few: at most 93 rows, with (longest) * rows a sixteenth of A's 144000 slots


@pytest.mark.parametrize("aat", [0, 1])
@pytest.mark.parametrize("listed", [1, 5, 11, 13, 40])
@pytest.mark.parametrize("block", [False, True])
def test_rows_of_both_sides(gpu, aat, listed, block):
    """Rows past the numeric tables (4096 values of C)."""
    wide = (np.arange(listed) * 8 * (1500 // listed)).astype(int)
    a = with_wide_rows(N, 12, np.r_[wide, wide + 3] if block else wide, 700, 5 * listed + aat, block)
    pa = gpu.prepare_identity_a(a)
    ref = oracle.spgemm(as_tuple(a), as_tuple(gpu.csr_transpose(a) if aat else a))
    pb = None
    for _ in range(2):
        pb = gpu.rebuild_b(pa, aat, pb)
        tc, st = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path="vector"))
        check_c(gpu, tc, ref)
    assert st["heavy_rows"] > 0


@pytest.mark.parametrize("path", ["vector", "auto", "tile"])
@pytest.mark.parametrize("aat", [0, 1])
def test_rows_beyond_the_symbolic_table(gpu, aat, path):
    """More than 768 C tiles in one row, and a hub that selects every row of B."""
    n = 8 * 1500
    a = with_wide_rows(n, 2, [4000], 900, 3 + aat)
    hub = with_wide_rows(n, 2, [17, 9000], n, 7 + aat)
    for x in (a, hub):
        pa = gpu.prepare_identity_a(x)
        ref = oracle.spgemm(as_tuple(x), as_tuple(gpu.csr_transpose(x) if aat else x))
        pb = None
        for _ in range(2):
            pb = gpu.rebuild_b(pa, aat, pb)
            tc, _ = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path=path))
            check_c(gpu, tc, ref)


def test_independent_b_and_new_values(gpu):
    """Another call may list other rows: B's wide rows change with its values
    kept, then its values with its structure kept."""
    n = 8 * 700
    a = with_wide_rows(n, 6, [800, 4000], 500, 11)
    pa = gpu.prepare_identity_a(a)
    pb = None
    sched = gpu.schedule(numeric_path="vector")
    for seed, wide in ((1, []), (2, np.arange(0, n, 16)), (3, [7])):
        b = with_wide_rows(n, 3, wide, 300, seed)
        src = gpu.upload_csr(b)
        pb = gpu.rebuild_b_general(pa, src, pb)
        tc, _ = gpu.tilespgemm(pa, pb, sched)
        check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(b)))
        b.val = np.random.default_rng(seed).uniform(-1, 1, b.nnz)
        src.set_values(b.val)
        gpu.update_b_values(pa, src, pb)
        tc, _ = gpu.tilespgemm(pa, pb, sched)
        check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(b)))


@pytest.mark.parametrize("aat", [0, 1])
def test_one_wide_row_takes_little_memory(gpu, aat):
    """One wide row in 262144 (A of 6.9e6 entries): with 12 bytes for every entry
    of B, 5 for every one of A and, for B = A^T, a second copy of B, it took 120
    to 200 MB; the row itself and what it selects take less than 1."""
    runtime = ctypes.CDLL("libamdhip64.so.7")   # the one the library has loaded

    def free():
        gpu.load().rtt_sync()
        free_bytes, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert runtime.hipMemGetInfo(ctypes.byref(free_bytes), ctypes.byref(total)) == 0
        return free_bytes.value

    def used(a):
        before = free()
        pa = gpu.prepare_identity_a(a)
        pb = None
        for _ in range(2):
            pb = gpu.rebuild_b(pa, aat, pb)
            gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path="vector", materialize_output=False))
        return before - free()

    a = gpu.gen_stencil27(64, 0.5, 1.5, 3)
    rng = np.random.default_rng(4)
    rows = np.r_[np.repeat(np.arange(a.m), np.diff(a.rowptr)), np.full(200, 5000)]
    cols = np.r_[a.col, rng.choice(a.n, 200, replace=False)]
    key, first = np.unique(rows.astype(np.int64) * a.n + cols, return_index=True)
    val = np.r_[a.val, np.ones(200)][first]
    wide = csr_from(a.m, a.n, key // a.n, key % a.n, val)
    used(a)   # what the library loads once
    plain = used(a)
    assert used(wide) - plain < 40 << 20
