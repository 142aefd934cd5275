"""The decode plan's rules follow the kernel that runs: 4 query heads per KV
head at head_dim 64 run on the vector units, 3 workgroups to a CU."""
import numpy as np
import pytest

from kunserve_amd import DecodePlan


@pytest.mark.parametrize("head_dim,ratio,per_cu", [
    (64, 4, 3), (64, 3, 2), (64, 1, 3), (128, 4, 2), (128, 2, 3), (256, 4, 1), (256, 1, 1)])
def test_how_many_workgroups_are_counted(head_dim, ratio, per_cu):
    """Rows of two partitions of 256 with 1 KV head."""
    for rows, counted in ((per_cu * 128, True), (per_cu * 128 + 1, False)):
        plan = DecodePlan([257] * rows, ratio, 1, None, part_tokens=256, num_cus=256,
                          upload=False, head_dim=head_dim)
        assert plan.info.num_merge == rows
        assert plan.num_counters == (plan.info.num_slots if counted else 0)


@pytest.mark.parametrize("rows,lo,hi,hq,hkv,part", [
    (48, 256, 4096, 16, 4, 1024),     # whole rows: 44.4 us a layer against 28.2
    (28, 241, 7578, 32, 8, 2048), (28, 241, 7578, 16, 4, 1024), (48, 256, 4096, 32, 8, 4096)])
def test_partition_length_at_head_dim_64(rows, lo, hi, hq, hkv, part):
    kv = np.random.default_rng(rows + hi).integers(lo, hi + 1, size=rows)
    plan = DecodePlan(kv, hq, hkv, None, num_cus=256, upload=False, head_dim=64)
    assert plan.info.part_tokens == part
