"""B's packed values for tiles of 1 to 32 entries, sparse and dense (24 entries
and more), by four lanes of a tile, and by one where most hold one entry:
products through them, and through a values-only update of the same
structure."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("singles", [0, 500])
@pytest.mark.parametrize("threshold", [24, 32])
def test_tiles_of_every_count(gpu, threshold, singles):
    rng = np.random.default_rng(threshold)
    k, n = 4 * 32, 8 * (40 + singles)
    cells = []
    for t in range(32):
        for j in range(6):   # tile (t, 5 j + t % 5) of t + 1 entries
            for p in rng.choice(32, t + 1, replace=False):
                cells.append((4 * t + p % 4, 8 * (5 * j + t % 5) + p // 4))
        cells += [(4 * t + int(j) % 4, 8 * (40 + int(j))) for j in range(singles)]
    cells = sorted(cells)
    r, c = np.array(cells).T
    b = csr_from(k, n, r, c, rng.uniform(-1, 1, len(r)))
    a = gpu.gen_random(300, k, 6, 3)
    pa = gpu.prepare_identity_a(a, dense_threshold=threshold)
    src = gpu.upload_csr(b)
    pb = gpu.rebuild_b_general(pa, src)
    sched = gpu.schedule(numeric_path="vector")
    tc, _ = gpu.tilespgemm(pa, pb, sched)
    check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(b)))
    b2 = csr_from(k, n, r, c, rng.uniform(-1, 1, len(r)))
    src.set_values(b2.val)
    gpu.update_b_values(pa, src, pb, "safe-auto")
    tc, _ = gpu.tilespgemm(pa, pb, sched)
    check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(b2)))
