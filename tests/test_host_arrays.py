"""Host arrays handed out by the library: they live as long as any view of
them, and tile-to-CSR conversion drops what lies outside the matrix in ragged
tiles and keeps everything in whole ones."""
import gc

import numpy as np
import pytest

import oracle
import rtt_amd as rt
from test_gpu_parity import as_tuple, check_c, csr_from


def random_tilec(m, n, seed, stray):
    """A TileC of random tiles over m x n, with entries beyond n in the last
    tile column and, with `stray`, local columns of 8 and more."""
    rng = np.random.default_rng(seed)
    tm, tn = -(-m // 8), -(-n // 8)
    ptr, cols, nnz, rp, lc, dense = [0], [], [0], [], [], {}
    for tr in range(tm):
        picks = np.sort(rng.choice(tn, min(tn, 3), replace=False))
        for tc in picks:
            count = 0
            for lr in range(8):
                rp.append(count)
                if tr * 8 + lr >= m:
                    continue
                for c in range(8):
                    if rng.random() < 0.4:
                        local = c + 8 if stray and rng.random() < 0.1 else c
                        lc.append(local)
                        if local < 8 and tc * 8 + local < n:
                            dense[(tr * 8 + lr, int(tc) * 8 + local)] = len(lc)
                        count += 1
            cols.append(tc)
            nnz.append(nnz[-1] + count)
        ptr.append(len(cols))
    tc = rt.TileC(m, n, tm, tn, len(cols), nnz[-1], np.array(ptr, np.int32),
                  np.array(cols, np.int32), np.array(nnz, np.int32), np.array(rp, np.uint8),
                  np.array(lc, np.uint8), np.arange(1.0, nnz[-1] + 1.0))
    return tc, dense


@pytest.mark.parametrize("m,n", [(1, 1), (8, 8), (40, 31), (37, 64), (65, 9)])
@pytest.mark.parametrize("stray", [False, True])
def test_tile2csr(m, n, stray):
    tc, want = random_tilec(m, n, m * 100 + n, stray)
    perm = np.random.default_rng(m).permutation(m).astype(np.int32)
    for got, order in ((rt.tile2csr(tc), np.arange(m)),
                       (rt.tile2csr_restore_rows(tc, perm, m), perm)):
        have = {(r, int(got.col[i])): got.val[i] for r in range(m)
                for i in range(got.rowptr[r], got.rowptr[r + 1])}
        assert have == {(int(order[r]), c): v for (r, c), v in want.items()}


def test_arrays_outlive_their_struct():
    tc, want = random_tilec(4000, 4000, 1, False)
    got = rt.tile2csr(tc)
    values, total = got.val, got.val.sum()
    del got
    gc.collect()
    again = [rt.tile2csr(tc) for _ in range(3)]      # would reuse freed memory
    values[0] += 1.0                                 # and stays writable
    assert values.sum() == total + 1.0 and len(values) == len(want)
    assert all(a.val.sum() == total for a in again)


@pytest.mark.gpu
@pytest.mark.parametrize("width", [3, 151])
def test_export(gpu, width):
    """C of less than one staging piece, and of more than the ring holds (40000
    rows of 301 entries, 96 MB of values), twice on one handle."""
    n = 40003
    rng = np.random.default_rng(width)
    rows = np.repeat(np.arange(n), width)
    cols = rows + np.tile(np.arange(width) - width // 2, n)
    keep = (cols >= 0) & (cols < n)
    a = csr_from(n, n, rows[keep], cols[keep], rng.uniform(-1, 1, int(keep.sum())))
    pa = gpu.prepare_identity_a(a)
    want = oracle.spgemm(as_tuple(a), as_tuple(a))
    first, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0))
    second, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0))
    check_c(gpu, first, want)
    check_c(gpu, second, want)
