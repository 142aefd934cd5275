"""kunserve_prefill_plan_packed: the query heads of a KV head share a tile
(row i of KV head g is token i / ratio of head g * ratio + i % ratio). Every
packed row of every KV head attends exactly the KV range its tile needs."""
import ctypes

import numpy as np
import pytest

from kunserve_amd import _lib


def _plan(name, q_lens, kv, hq, hkv, num_cus=256, head_dim=128):
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    kv = np.asarray(kv, dtype=np.int32)
    cap = _lib.lib().kunserve_prefill_plan_bound(qi.ctypes.data, len(kv), hq, head_dim)
    buf = np.zeros(cap, dtype=np.int32)
    info = _lib.PrefillPlanInfo()
    _lib.call(name, qi.ctypes.data, kv.ctypes.data, len(kv), hq, hkv, head_dim, num_cus,
              buf.ctypes.data, cap, ctypes.byref(info))
    return (info, buf[:6 * info.num_tiles].reshape(-1, 6),
            buf[6 * info.num_tiles:info.plan_ints].reshape(-1, 5))


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("num_cus", [1, 256, 2048])
@pytest.mark.parametrize("hq,hkv", [(8, 4), (12, 4), (32, 8), (35, 5), (16, 1), (64, 2)])
def test_packed_plan_covers_every_row_once(hq, hkv, num_cus, head_dim):
    rng = np.random.default_rng(hq + hkv + num_cus)
    ratio = hq // hkv
    q_lens = np.r_[rng.integers(0, 700, 4), 1, 0, 64, 65, 256 // ratio, 256 // ratio + 1]
    kv = q_lens + np.r_[rng.integers(0, 3000, 4), 4000, 5, 0, 1, 63, 64]
    info, items, merges = _plan("kunserve_prefill_plan_packed", q_lens, kv, hq, hkv, num_cus,
                                head_dim)
    tq = info.tile_q
    real = items[items[:, 0] >= 0]
    ranges = {}
    for b, r0, h, lo, hi, slot in real.tolist():
        ranges.setdefault((b, r0, h), []).append((lo, hi, slot))
    assert set(ranges) == {(b, r0, ~g) for b in range(len(kv))
                           for r0 in range(0, int(q_lens[b]) * ratio, tq) for g in range(hkv)}
    merged = {(b, r0, h): (s0, n) for b, r0, h, s0, n in merges.tolist()}
    slots = []
    for (b, r0, h), rs in ranges.items():
        last_token = (min(r0 + tq, int(q_lens[b]) * ratio) - 1) // ratio
        rs.sort()
        assert rs[0][0] == 0 and rs[-1][1] == kv[b] - q_lens[b] + last_token + 1
        assert all(x[1] == y[0] and x[1] % 64 == 0 for x, y in zip(rs, rs[1:]))
        if len(rs) == 1:
            assert rs[0][2] == -1 and (b, r0, h) not in merged
        else:
            s0, n = merged[(b, r0, h)]
            assert n == len(rs) and [r[2] for r in rs] == list(range(s0, s0 + n))
            slots += [r[2] for r in rs]
    assert sorted(slots) == list(range(info.num_slots)) and len(merged) == info.num_merge


def test_packed_plan_without_gqa_is_the_plain_plan():
    args = ([300, 1, 512], [900, 70, 512], 4, 4)
    plain = _plan("kunserve_prefill_plan", *args)
    packed = _plan("kunserve_prefill_plan_packed", *args)
    assert np.array_equal(plain[1], packed[1]) and np.array_equal(plain[2], packed[2])


def test_packed_plan_rejects_rows_too_long_to_number():
    with pytest.raises(_lib.KunserveError, match="too long"):
        qi = np.array([0, 2**28], dtype=np.int32)
        kv = np.array([2**28], dtype=np.int32)
        buf = np.zeros(64, dtype=np.int32)
        _lib.call("kunserve_prefill_plan_packed", qi.ctypes.data, kv.ctypes.data, 1, 8, 1, 128,
                  256, buf.ctypes.data, 64, ctypes.byref(_lib.PrefillPlanInfo()))
    _plan("kunserve_prefill_plan_packed", [4], [4], 8, 1)
