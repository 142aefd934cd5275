"""Split prefill plans: how long the pieces are and where they go."""
import heapq

import numpy as np
import pytest

from kunserve_amd import PrefillPlan


def _plan(rows, hq, hkv, head_dim):
    q = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    plan = PrefillPlan(np.concatenate([[0], np.cumsum(q)]), kv, hq, hkv, None, num_cus=256,
                       upload=False, head_dim=head_dim)
    return plan, plan.plan_host[:6 * plan.info.num_tiles].reshape(-1, 6)


@pytest.mark.parametrize("rows,hq,hkv,head_dim,tiles,pieces", [
    ([(512, 130), (512, 130)], 32, 8, 128, 5, 240),   # 288 of 4 by the CUs' mean load
    ([(415, 7939)], 64, 8, 64, 64, 256),              # 312 of 53: the last start at 56 tiles
    ([(1212, 143), (1212, 143)], 16, 8, 128, 11, None)])
def test_chunk_leaves_one_piece_per_cu(rows, hq, hkv, head_dim, tiles, pieces):
    plan, work = _plan(rows, hq, hkv, head_dim)
    assert plan.info.kv_chunk == 64 * tiles
    n = int((work[:, 0] >= 0).sum())
    assert n == pieces if pieces else n <= 256


@pytest.mark.parametrize("rows,hq,hkv,head_dim", [
    ([(314, 8433)], 16, 4, 128), ([(394, 332)], 32, 4, 256), ([(57, 17982), (57, 900)], 8, 2, 256),
    ([(31, 9031), (3, 50), (8, 700), (20, 100)], 8, 2, 128), ([(100, 50)], 4, 4, 128)])
def test_one_round_fits_every_xcd(rows, hq, hkv, head_dim):
    """Pieces that fit the 256 CUs: no XCD has more than its 32."""
    plan, work = _plan(rows, hq, hkv, head_dim)
    assert 0 < (work[:, 0] >= 0).sum() <= 256
    assert max(int((work[x::8, 0] >= 0).sum()) for x in range(8)) <= 32


@pytest.mark.parametrize("rows,hq,hkv,head_dim,splits", [
    ([(64, 576)], 16, 4, 128, True), ([(64, 512)], 16, 4, 128, False),    # 10 and 9 tiles
    ([(300, 40), (17, 9)], 8, 8, 128, False), ([(1, 255)], 8, 8, 64, False),
    ([(78, 326)] * 9, 16, 4, 128, False), ([(1, 639)], 32, 8, 256, True)])
def test_splits_shorten_the_longest_item(rows, hq, hkv, head_dim, splits):
    plan, work = _plan(rows, hq, hkv, head_dim)
    assert (plan.info.num_merge > 0) == splits
    if not splits:   # every item whole, and still at most 32 to an XCD
        assert (work[work[:, 0] >= 0, 5] == -1).all() and (work[work[:, 0] >= 0, 3] == 0).all()
        assert max(int((work[x::8, 0] >= 0).sum()) for x in range(8)) <= 32


@pytest.mark.parametrize("rows,hq,hkv,counted", [
    ([(300, 600)], 8, 8, True), ([(300, 600)] * 2, 8, 8, False),      # 64 and 128 slots
    ([(300, 600)] * 2, 8, 2, True), ([(515, 12698)], 64, 8, True), ([(416, 500)], 4, 4, True),
    ([(300, 8000)], 8, 2, False)])                                     # more than 4 splits
def test_who_combines_the_splits(rows, hq, hkv, counted):
    """The launch, up to 4 splits; without GQA up to 64 slots of partials."""
    plan, _ = _plan(rows, hq, hkv, 128)
    assert plan.info.num_merge > 0
    assert plan.num_counters == (8 * plan.info.num_slots if counted else 0)


@pytest.mark.parametrize("rows,hq,hkv,head_dim,tiles", [
    ([(515, 12698)], 64, 8, 128, None), ([(456, 18222)], 48, 8, 256, None),
    ([(512, 130), (512, 130)], 32, 8, 128, 5), ([(416, 2893)] * 4, 32, 8, 128, None)])
def test_two_rounds_end_near_the_mean(rows, hq, hkv, head_dim, tiles):
    """Pieces taken longest first by 256 CUs (a start counting 3.5 tiles) end at
    most a quarter after the CUs' mean load."""
    plan, work = _plan(rows, hq, hkv, head_dim)
    if tiles:
        assert plan.info.kv_chunk == 64 * tiles
        return
    work = work[work[:, 0] >= 0]
    costs = sorted((work[:, 4] + 63) // 64 - work[:, 3] // 64 + 3.5, reverse=True)
    ends = [0.0] * 256
    heapq.heapify(ends)
    for c in costs:
        heapq.heapreplace(ends, ends[0] + c)
    assert max(ends) <= 1.25 * sum(costs) / 256
