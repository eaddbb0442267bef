"""Each array of a host result lives by itself: one kept small array does not
keep the large ones."""
import gc

import numpy as np

import rtt_amd as rt


def resident():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[1]) * 4096


def full_tiles(tm, tn):
    n = tm * tn
    return rt.TileC(8 * tm, 8 * tn, tm, tn, n, 64 * n,
                    (np.arange(tm + 1) * tn).astype(np.int32),
                    np.tile(np.arange(tn, dtype=np.int32), tm),
                    (np.arange(n + 1) * 64).astype(np.int32),
                    np.tile((np.arange(8) * 8).astype(np.uint8), n),
                    np.tile(np.arange(8, dtype=np.uint8), 8 * n), np.ones(64 * n))


def test_a_kept_array_keeps_only_itself():
    tc = full_tiles(400, 200)            # 5.1e6 entries: 61 MB of columns and values
    got = rt.tile2csr(tc)
    assert got.nnz == tc.nnz and got.val.sum() == tc.nnz
    rows, col = got.rowptr, got.col[:1000].copy()
    gc.collect()
    full = resident()
    del got
    gc.collect()
    assert full - resident() > 50 << 20, "columns and values are still there"
    assert np.array_equal(rows, np.arange(3201) * 1600) and col[999] == 999


def test_generated_matrices_too():
    a = rt.gen_random(200000, 1000, 25, 1)   # 60 MB
    val = a.val
    total = val.sum()
    gc.collect()
    full = resident()
    del a
    gc.collect()
    assert full - resident() > 15 << 20, "the columns are still there"
    val[0] += 1.0
    assert abs(val.sum() - total - 1.0) < 1e-6 and len(val) == 5_000_000
