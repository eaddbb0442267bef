"""Infinities, NaN, the type's extremes, subnormals and signed zeros through the
numeric kernels of every row class but the matrix cores': an entry of C is the
sum of its stored products and of nothing else (absent slots of dense tiles are
never multiplied), with the oracle's sums of the same products."""
import numpy as np
import pytest

import oracle
from test_gpu_few_slab_rows import with_wide_rows
from test_gpu_parity import as_tuple, csr_from
from test_gpu_slab_by_tiles import tiled

pytestmark = pytest.mark.gpu

SPECIAL = np.array([np.inf, -np.inf, np.nan, 1.7976931348623157e308, -1.7976931348623157e308,
                    5e-324, 2.2e-308, -0.0, 0.0])


def holes(n, seed):
    """Dense A and B tiles with absent slots beside sparse ones."""
    rng = np.random.default_rng(seed)
    d = rng.random((n, n)) < np.where(np.arange(n)[:, None] // 16 % 2 == 0, 0.9, 0.05)
    r, c = np.nonzero(d)
    return csr_from(n, n, r, c, rng.uniform(-1, 1, len(r)))


MATS = {
    "one wave": lambda g: g.gen_laplace2d(40, 0.1, 1),
    "sparse C tiles": lambda g: g.gen_stencil27(9, 0.5, 1.5, 2),
    "full C tiles": lambda g: g.gen_banded(2000, 12, 10, 3),
    "medium": lambda g: g.gen_banded(2000, 40, 30, 4),
    "large and beyond": lambda g: g.gen_banded(2500, 200, 60, 5),
    "dense tiles": lambda g: holes(96, 6),
    "many wide rows": lambda g: g.gen_rmat(10, 12, seed=7),
    "few wide rows": lambda g: with_wide_rows(8 * 1500, 12, [40, 9000], 700, 8),
    "wide rows by tiles": lambda g: tiled(8 * 400, 8 * 400, 8, 4,
                                          np.where(np.arange(400) % 40 == 3, 300, 12), 0.6, 9),
}


@pytest.mark.parametrize("aat", [0, 1])
@pytest.mark.parametrize("name", list(MATS))
def test_special_values(gpu, name, aat):
    a = MATS[name](gpu)
    rng = np.random.default_rng(11)
    at = rng.choice(a.nnz, max(12, a.nnz // 400), replace=False)
    a.val = np.array(a.val)
    a.val[at] = SPECIAL[rng.integers(0, len(SPECIAL), len(at))]
    pa = gpu.prepare_identity_a(a)
    b = gpu.csr_transpose(a) if aat else a
    with np.errstate(all="ignore"):
        ref = oracle.spgemm(as_tuple(a), as_tuple(b))
        absa = gpu.CsrMatrix(a.m, a.n, a.rowptr, a.col, np.abs(a.val))
        absb = gpu.csr_transpose(absa) if aat else absa
        bound = oracle.spgemm(as_tuple(absa), as_tuple(absb))["val"]
    pb = None
    for _ in range(2):
        pb = gpu.rebuild_b(pa, aat, pb)
        tc, _ = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path="vector"))
        got = gpu.tile2csr(tc)
        assert np.array_equal(got.col, ref["col"])
        assert np.array_equal(got.rowptr.astype(np.int64), ref["rowptr"])
        want = ref["val"]
        # Without a special value or an overflow among its products: the
        # forward bound of two sums of at most 4096, and a subnormal's spacing a
        # product.  With one the sum is not finite in any order.
        fin = np.isfinite(bound)
        err = np.abs(got.val[fin] - want[fin])
        assert np.all(err <= 2 * 4096 * 2.0 ** -53 * bound[fin] + 4096 * 5e-324)
        assert not np.any(np.isfinite(got.val[~np.isfinite(want)]))
        assert 0 < np.count_nonzero(~np.isfinite(want)) < want.size
