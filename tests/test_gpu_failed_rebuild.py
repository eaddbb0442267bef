"""A rebuild that is refused for its size leaves a B that no call reads, and
that the next rebuild makes good."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import as_tuple, check_c, csr_from

pytestmark = pytest.mark.gpu

INVALID, OVERFLOW = 1, 3


def test_a_refused_rebuild_is_not_read(gpu):
    n = 4_400_000
    a = csr_from(8, n, [0, 3], [5, n - 1], [2.0, 3.0])
    pa = gpu.prepare_identity_a(a, 1)          # every tile dense: 32 slots each
    small = gpu.gen_random(n, 300, 1, 2)
    src = gpu.upload_csr(small)
    pb = gpu.rebuild_b_general(pa, src)
    pb.tiles()
    # 7e7 scattered entries: 2.2e9 slots, beyond the int32 tile ABI.
    with pytest.raises(gpu.RttError) as e:
        gpu.rebuild_b_general(pa, gpu.upload_csr(gpu.gen_random(n, 40_000_000, 16, 3)), pb)
    assert e.value.code == OVERFLOW
    for read in (pb.tiles, lambda: gpu.tilespgemm(pa, pb)):
        with pytest.raises(gpu.RttError) as e:
            read()
        assert e.value.code == INVALID
    pb = gpu.rebuild_b_general(pa, src, pb)
    tc, _ = gpu.tilespgemm(pa, pb)
    check_c(gpu, tc, oracle.spgemm(as_tuple(a), as_tuple(small)))
    assert np.diff(pb.tiles()["tile_row_ptr"]).sum() == pb.tiles()["num_tiles"]
