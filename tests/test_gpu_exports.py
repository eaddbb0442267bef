"""Exports of C to the host share one ring of pinned memory: many handles add
nothing to it, it is given back with the last of them, and handles may export
from several threads at once."""
import gc
import threading

import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c

pytestmark = pytest.mark.gpu


def pinned_bytes():
    """Host memory the process has mapped from the GPU driver, device memory
    apart: mappings of 8 MB and more (the ring's size) that are readable."""
    total = 0
    with open("/proc/self/smaps") as f:
        lines = f.read().split("\n")
    for line in lines:
        part = line.split()
        if len(part) >= 5 and "-" in part[0] and "rw" in part[1]:
            lo, hi = (int(x, 16) for x in part[0].split("-"))
            name = part[5] if len(part) > 5 else ""
            if name.startswith("/dev/") and hi - lo == 8 << 20:
                total += hi - lo
    return total


def test_many_handles_share_the_pinned_ring(gpu):
    a = gpu.gen_laplace2d(40, 0.1, 1)
    want = oracle.spgemm(as_tuple(a), as_tuple(a))
    gc.collect()
    held = []

    def export(n):
        for _ in range(n):
            pa = gpu.prepare_identity_a(a)
            pb = gpu.rebuild_b(pa, 0)
            tc, _ = gpu.tilespgemm(pa, pb)
            held.append((pa, pb))
        return tc

    check_c(gpu, export(1), want)
    one = pinned_bytes()
    check_c(gpu, export(24), want)
    assert pinned_bytes() <= one + (16 << 20), "a ring a handle would be 192 MB"
    held.clear()
    gc.collect()
    check_c(gpu, export(1), want)   # a ring anew after the last handle


def test_exports_from_threads(gpu):
    """Distinct handles in distinct threads, results of less and of more than a
    piece of the ring, and of more than all of it."""
    mats = [gpu.gen_laplace2d(20, 0.1, 1), gpu.gen_fem_blocks(2500, 6, True, 2),
            gpu.gen_random(3000, 3000, 30, 3), gpu.gen_banded(9000, 40, 20, 4)]
    sched = gpu.schedule(numeric_path="tile")   # the same bits every time
    first, errors = [], []
    for a in mats:
        pa = gpu.prepare_identity_a(a)
        tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0), sched)
        check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(a)))
        first.append(tc)

    def work(a, want):
        try:
            for _ in range(6):
                pa = gpu.prepare_identity_a(a)
                tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0), sched)
                assert np.array_equal(tc.tile_ptr, want.tile_ptr)
                assert np.array_equal(tc.tile_columnidx, want.tile_columnidx)
                assert np.array_equal(tc.tile_csr_Col, want.tile_csr_Col)
                assert np.array_equal(tc.tile_csr_Value, want.tile_csr_Value)
        except BaseException as e:   # noqa: B036 (reported by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=x) for x in zip(mats, first)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
