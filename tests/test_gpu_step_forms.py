"""Steps whose launches append, in the forms that move the appended row's
address: page sizes, ratios whose head groups share a KV head, k and v as
slices of one projection, rows with more pages than a workgroup stages, and
rows of many partitions. Pages hold the appended bytes, outputs match the
oracle on the pages after the append."""
import math

import numpy as np
import pytest
import torch

from kunserve_amd import AttentionStep
from oracle import paged_attention_ref as ref

from helpers import ATOL, ATOL_BF16, max_abs, random_pool, random_tensor, to_numpy


def _run(device, rows, hq, hkv, hd, ps, dtype=torch.float16):
    """rows: (new tokens, prefix, decodes). Runs layer 1 of 2 and checks it."""
    q_lens = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    need = [-(-n // ps) for n in kv]
    npg = sum(need) + 3
    perm = np.random.default_rng(hd + ps).permutation(npg).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    pool = random_pool(npg, 2, hkv, ps, hd, device, 3, dtype=dtype)
    first = [n if d else p for (_, p, d), n in zip(rows, kv)]
    step = AttentionStep(pool, hq, q_lens, first, [1 - r[2] for r in rows], tables)
    assert step._step.appends == 1
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, dtype=dtype)
    proj = random_tensor((T, 2 * hkv, hd), device, 5, dtype=dtype)
    k, v = proj[:, :hkv], proj[:, hkv:]
    kh, vh = to_numpy(pool.k), to_numpy(pool.v)
    out, again = step.run(1, q, k, v), step.run(1, q, k, v)
    torch.cuda.synchronize()
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    indices = np.array([p for t in tables for p in t], dtype=np.int32)
    lens = np.array(kv, dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    ref.append_kv(kh, vh, 1, indptr, indices, lens, qi, to_numpy(k), to_numpy(v))
    assert np.array_equal(to_numpy(pool.k), kh) and np.array_equal(to_numpy(pool.v), vh)
    want = ref.prefill_attention(to_numpy(q), qi, kh, vh, 1, indptr, indices, lens,
                                 1 / math.sqrt(hd))
    assert torch.equal(out, again)
    assert max_abs(out, want) <= (ATOL if dtype == torch.float16 else ATOL_BF16)
    return step


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (8, 2), (34, 2)])
@pytest.mark.parametrize("ps", [4, 256])
def test_decode_appends(device, hq, hkv, hd, ps, dtype):
    kv = [1, 4, 5, 256, 257, 700, 513, 2047]
    step = _run(device, [(1, n - 1, 1) for n in kv], hq, hkv, hd, ps, dtype)
    assert step.decode.plan.info.group_size == {1: 1, 4: 4, 17: 1}[hq // hkv]


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("split", [False, True])
def test_prefill_appends_without_staged_pages(device, monkeypatch, hd, split):
    """2087 pages of 4 tokens: more than a workgroup's page ids in LDS."""
    from kunserve_amd import paged_kv
    if not split:
        monkeypatch.setattr(paged_kv, "_num_cus", lambda d: 1)
    step = _run(device, [(45, 8301, 0), (3, 61, 0), (1, 99, 1)], 2, 1, hd, 4)
    info = step.prefill.plan.info
    assert info.max_kv_len > 4 * 2048 and (info.num_merge > 0) == split


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,hd", [(4, 1, 128), (2, 2, 64), (8, 1, 256)])
def test_decode_of_a_long_row(device, hq, hkv, hd):
    step = _run(device, [(1, 99999, 1), (1, 299, 1), (1, 32767, 1)], hq, hkv, hd, 16)
    info = step.decode.plan.info
    assert info.num_merge >= 2 and step._step.num_counters == 0
    assert -(-100000 // info.part_tokens) > 8
