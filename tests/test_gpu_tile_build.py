"""The CSR -> tile builder at its edges, bit for bit against the oracle's
tiles: workgroup boundaries (128 B tile rows, 64 A tile rows), rows at and past
the limit of the merge (128 entries a scalar row on average over a tile row),
long rows over several column windows (4096 tile columns), duplicates in both,
rows past the column stage, and rebuilds of one handle from other operands."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_a_tiles, csr_from, oracle_tiles_equal, sub_rows

pytestmark = pytest.mark.gpu


def matrix(m, n, lengths, seed, dups=0, spread=None):
    """m x n CSR with lengths[i] entries in row i, the first `dups` of a row
    twice; columns from the first `spread` (all by default)."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(m):
        c = np.sort(rng.choice(spread or n, size=lengths[i], replace=False))
        c = np.sort(np.concatenate([c, c[:dups], c[:dups]])) if dups else c
        rows.append(np.full(len(c), i))
        cols.append(c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    return csr_from(m, n, rows, cols, rng.uniform(-1, 1, len(rows)))


def check_b(rt, pa, pb, b, threshold=24):
    ai = pa.info()[1]
    want = oracle.hybrid_tiles(*sub_rows(as_tuple(b), ai), 4, 8, True, threshold, build_csc=True)
    oracle_tiles_equal(pb.tiles(), want, csc=True)


CASES = {
    # name: (rows, columns, entries per row, duplicates, column range)
    "half a workgroup": (256, 300, lambda i: 3, 0, None),
    "one workgroup": (512, 300, lambda i: 3, 0, None),
    "one row past a workgroup": (513, 300, lambda i: 3 + i % 5, 0, None),
    "at the limit": (40, 900, lambda i: 128, 0, None),
    "just past the limit": (40, 900, lambda i: 129 if i < 4 else 2, 0, None),
    "long and short mixed": (600, 4000, lambda i: 900 if i % 97 == 5 else i % 7, 0, None),
    "long over windows": (64, 70000, lambda i: 2500 if i % 16 == 3 else 1, 0, None),
    "dense rows": (48, 260, lambda i: 250, 0, None),
    "duplicates in short rows": (300, 200, lambda i: i % 12, 5, None),
    "duplicates in long rows": (36, 1500, lambda i: 400 if i < 8 else 4, 7, None),
    "duplicates filling tiles": (40, 64, lambda i: 8, 8, 8),
    "past the stage": (1024, 400, lambda i: 120 if i < 512 else 0, 0, None),
    "past the largest stage": (512, 400, lambda i: 126 if i < 300 else 3, 0, None),
    "empty rows": (520, 90, lambda i: 4 if 250 < i < 262 else 0, 0, None),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("threshold", [24, 1])
def test_tiles_match_the_oracle(gpu, name, threshold):
    m, n, f, dups, spread = CASES[name]
    b = matrix(m, n, [f(i) for i in range(m)], 5, dups, spread)
    pb_a = gpu.prepare_identity_a(b, threshold)      # as A: 8x4 tiles
    check_a_tiles(gpu, b, pb_a, threshold)
    a = gpu.gen_random(50, m, min(m, 9), 3)          # as B: 4x8 tiles
    pa = gpu.prepare_identity_a(a, threshold)
    src = gpu.upload_csr(b)
    pb = gpu.rebuild_b_general(pa, src)
    check_b(gpu, pa, pb, b, threshold)
    # In place, then new values by the source map: a rebuild's payload.
    pb = gpu.rebuild_b_general(pa, src, pb)
    check_b(gpu, pa, pb, b, threshold)
    b.val = np.random.default_rng(9).uniform(-1, 1, b.nnz)
    src.set_values(b.val)
    gpu.update_b_values(pa, src, pb)
    check_b(gpu, pa, pb, b, threshold)


def test_one_handle_over_operands_of_other_sizes(gpu):
    """A handle that shrinks and grows again, and long rows through an order."""
    a = gpu.gen_random(60, 400, 8, 1)
    pa = gpu.prepare_identity_a(a)
    pb = None
    for seed, per in ((1, 5), (2, 90), (3, 1), (4, 300)):
        b = matrix(400, 3000, [per] * 400, seed)
        pb = gpu.rebuild_b_general(pa, gpu.upload_csr(b), pb)
        check_b(gpu, pa, pb, b)
    rng = np.random.default_rng(8)
    order = rng.permutation(400).astype(np.int32)
    px = gpu.prepare_external_a(a, np.arange(60, dtype=np.int32), order)
    px_b = gpu.rebuild_b_general(px, gpu.upload_csr(b))
    mapped = b.to_scipy()[order]
    mapped.sort_indices()
    check_b(gpu, px, px_b, gpu.CsrMatrix(400, 3000, mapped.indptr.astype(np.int32),
                                         mapped.indices.astype(np.int32), mapped.data))
