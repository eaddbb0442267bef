"""Split-precision batches: C tiles of 1 to 17 pairs (batches of 8 and their
remainders), and operands whose magnitudes span 0 to 40 binades per tile row,
around the 20 at which a batch leaves the slices, with zeros, negative values
and subnormals, against the form's own error bound."""
import numpy as np
import pytest

from test_gpu_parity import csr_from, oracle_product
from test_gpu_tile import split_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs", [1, 2, 3, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("span", [0, 11, 12, 19, 20, 21, 40])
def test_pairs_and_spans(gpu, pairs, span):
    """One block of `pairs` A tiles across, squared: every C tile sums `pairs`
    products."""
    rng = np.random.default_rng(pairs * 100 + span)
    n = 4 * pairs
    full = rng.uniform(0.5, 1.0, (n, n)) * rng.choice([-1.0, 1.0], (n, n))
    full *= 2.0 ** -rng.integers(0, span + 1, (n, n))
    keep = rng.random((n, n)) < 0.8
    keep[:, 0] = keep[0, :] = True
    r, c = np.nonzero(keep)
    v = full[r, c]
    v[rng.random(len(v)) < 0.05] = 0.0      # stored zeros
    a = csr_from(n, n, r, c, v)
    if span <= 20:
        split_run(gpu, a, 0)
        return
    # Batches past the span are FP64 sums of 4 products a pair, which may lose
    # half an ulp of the sum of magnitudes at each step; those within it have
    # the slices' error, at most 2^-61 of a row's (column's) maximum per entry.
    pa = gpu.prepare_identity_a(a)
    tc, _ = gpu.tilespgemm(pa, gpu.rebuild_b(pa, 0), gpu.schedule(precision="split-bf16"))
    ref = oracle_product(a, 0)
    csr = gpu.tile2csr(tc)
    d = abs(a.to_scipy().toarray())
    some = (d > 0).astype(float)
    some[r, c] = 1.0
    slices = d.max(axis=1)[:, None] * (some @ d) + (d @ some) * d.max(axis=0)[None, :]
    bound = 2.0 ** -61 * slices + 4 * pairs * 2.0 ** -53 * (d @ d)
    rows = np.repeat(np.arange(n), np.diff(csr.rowptr))
    err = np.abs((csr.val - ref["hi"]) - ref["lo"])
    assert np.array_equal(csr.col, ref["col"])
    assert np.all(err <= bound[rows, csr.col])


@pytest.mark.parametrize("scale", [2.0 ** -530, 2.0 ** 500])
def test_scales(gpu, scale):
    """Products near the ends of the range: C of 2^-1060 (subnormal, so the
    bound's FP64 rounding does not hold there: compared with the FP64 form to
    within a few of the smallest subnormals) and of 2^1000."""
    rng = np.random.default_rng(7)
    n = 24
    r, c = np.nonzero(rng.random((n, n)) < 0.7)
    a = csr_from(n, n, r, c, rng.uniform(-1, 1, len(r)) * scale)
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b(pa, 0)
    got, _ = gpu.tilespgemm(pa, pb, gpu.schedule(precision="split-bf16"))
    want, _ = gpu.tilespgemm(pa, pb, gpu.schedule(numeric_path="tile"))
    g, w = got.tile_csr_Value, want.tile_csr_Value
    # 24 products of at most scale^2, rounded differently: 24 * 2^-50 of them,
    # and 24 roundings to a multiple of 2^-1074
    assert np.all(np.abs(g - w) <= 24 * 2.0 ** -50 * scale * scale + 24 * 2.0 ** -1074)
