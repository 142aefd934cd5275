"""Decode with all query heads of a KV head in one workgroup (2 to 16 MFMA
columns, head_dim 64, 128 and 256): ratios that are and are not powers of
two, rows that end at and beside step and wave boundaries, whole and split
rows, and a page id outside the pool, against the oracle. The
probabilities enter the matrix unit as two 16-bit terms, so the result is
off by the output's rounding (u |x|, u = 2^-11 with the 11 significant bits of
fp16 and 2^-8 with the 8 of bf16) and by
what the terms leave: 2^-17 of a weighted mean of |v| < 5 in bf16, and fp32
sums, together below 1e-4."""
import ctypes
import math

import numpy as np
import pytest
import torch

from kunserve_amd import DecodePlan, _lib, paged_decode
from oracle import paged_attention_ref as ref

from helpers import compact_for_oracle, random_pool, random_tensor, table_from_csr, to_numpy


def grouped_plan(kv, hq, hkv, part=0, num_cus=256):
    kv = np.asarray(kv, dtype=np.int32)
    cap = _lib.lib().kunserve_decode_plan_bound(kv.ctypes.data, kv.size)
    buf = np.zeros(cap, dtype=np.int32)
    info = _lib.DecodePlanInfo()
    _lib.call("kunserve_decode_plan_grouped", kv.ctypes.data, kv.size, hq, hkv, 128, num_cus, part,
              buf.ctypes.data, cap, ctypes.byref(info))
    return info, buf[:4 * info.num_work].reshape(-1, 4)


@pytest.mark.parametrize("ratio,group", [(1, 1), (2, 2), (3, 3), (7, 7), (8, 8), (12, 12),
                                         (16, 16), (17, 1), (24, 12), (32, 16)])
def test_grouped_plan_takes_the_largest_divisor(ratio, group):
    kv = [5000, 0, 17, 300, 4096]
    info, work = grouped_plan(kv, 2 * ratio, 2)
    assert info.group_size == group
    covered = np.zeros(len(kv), dtype=np.int64)
    for seq, b, e, _ in work[work[:, 0] >= 0].tolist():
        covered[seq] += e - b
    assert covered.tolist() == kv


@pytest.mark.parametrize("kv,hq,hkv,head_dim,part", [
    ([777], 32, 8, 128, 128),                       # one row: many short partitions
    ([777] * 64, 32, 8, 128, 1024),                 # whole rows fill the device
    ([512] * 8, 32, 32, 128, 512),
    ([8000] * 128, 32, 8, 128, 4096),
    ([20000], 8, 1, 128, 256),
    ([1584] * 28, 32, 8, 256, 2048),
    ([1], 4, 4, 64, 128), ([], 4, 4, 64, 128), ([233, 233], 40, 8, 128, 256)])
def test_grouped_plan_partition(kv, hq, hkv, head_dim, part):
    kv = np.asarray(kv, dtype=np.int32)
    plan = DecodePlan(kv, hq, hkv, None, num_cus=256, upload=False, head_dim=head_dim)
    assert plan.info.part_tokens == part
    # combined by the launch: one round of workgroups, at most 8 partitions a row
    parts = -(-kv // part)
    groups = hq // plan.info.group_size
    counted = (plan.info.num_merge > 0 and parts.max(initial=0) <= 8
               and parts.sum() * groups <= 256 * (2 if plan.info.group_size > 2 else 4))
    assert plan.num_counters == (plan.info.num_slots * groups if counted else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("ratio,hkv", [(2, 3), (3, 2), (4, 2), (5, 1), (7, 2), (8, 1), (12, 1),
                                       (16, 1), (32, 1)])
def test_grouped_decode_matches_the_oracle(device, ratio, hkv, head_dim, dtype):
    rng = np.random.default_rng(ratio * head_dim)
    kv = np.array([1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513,
                   1500, 0], dtype=np.int32)
    need = (kv + 15) // 16
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    npg = int(indptr[-1]) + 3
    indices = rng.permutation(npg)[:indptr[-1]].astype(np.int32)
    hq = ratio * hkv
    pool = random_pool(npg, 1, hkv, 16, head_dim, device, 5, dtype=dtype)
    q = random_tensor((len(kv), hq, head_dim), device, 6, 2.0, dtype=dtype)
    table = table_from_csr(indptr, indices, kv, device)
    k, v, ip, ix = compact_for_oracle(pool, 0, indptr, indices)
    want = ref.decode_attention(to_numpy(q), k, v, 0, ip, ix, kv, 1 / math.sqrt(head_dim))
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for part in (0, 256, 4096):
        plan = DecodePlan(kv, hq, hkv, device, part_tokens=part)
        assert plan.info.group_size == (16 if ratio == 32 else ratio)
        out = to_numpy(paged_decode(pool, 0, table, q, plan)).astype(np.float64)
        off = np.abs(out - want) - 1.001 * u * np.abs(want)
        assert off.max() <= 1e-4, (part, off.max())


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("ratio", [3, 8])
def test_grouped_decode_drops_pages_outside_the_pool(device, head_dim, ratio):
    """Tokens of a page id outside the pool leave the softmax: the result is
    that of the row without the page."""
    kv, ps, hkv = 200, 16, 2
    pool = random_pool(20, 1, hkv, ps, head_dim, device, 7)
    q = random_tensor((1, ratio * hkv, head_dim), device, 8)
    ids = np.arange(13, dtype=np.int32)
    bad = ids.copy()
    bad[4] = 20
    good = np.delete(ids, 4)
    outs = []
    for pages, n in ((bad, kv), (good, kv - ps)):
        lens = np.array([n], dtype=np.int32)
        table = table_from_csr(np.array([0, len(pages)], np.int32), pages, lens, device)
        outs.append(paged_decode(pool, 0, table, q, DecodePlan(lens, ratio * hkv, hkv, device)))
    torch.cuda.synchronize()
    assert (outs[0].float() - outs[1].float()).abs().max().item() <= 2e-3
