"""The tail records are the last call's: none after a call without a tail queue."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other", [{"numeric_path": "vector"},
                                   {"numeric_path": "tile", "lb_mode": "static"},
                                   {"numeric_path": "tile", "split_threshold": 1e9}])
def test_records_of_the_last_call(gpu, other):
    a = gpu.gen_fem_blocks(400, 6, True, 31)
    pa = gpu.prepare_identity_a(a)
    pb = gpu.rebuild_b(pa, 0)
    split = gpu.schedule(materialize_output=False, numeric_path="tile", split_threshold=40.0,
                         split_chunk_target=20.0, force_tail_split=1)
    _, st = gpu.tilespgemm(pa, pb, split)
    assert len(gpu.last_tail_records(pa)["task"]) == st["tail_records"] > 0
    _, st = gpu.tilespgemm(pa, pb, gpu.schedule(materialize_output=False, **other))
    assert st["tail_records"] == 0 == len(gpu.last_tail_records(pa)["task"])
    _, st = gpu.tilespgemm(pa, pb, split)
    assert len(gpu.last_tail_records(pa)["task"]) == st["tail_records"] > 0
