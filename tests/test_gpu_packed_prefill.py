"""Prefill on packed plans (the query heads of a KV head share a tile):
ratios that divide a tile and ratios that do not, rows that end at and
beside tile edges, whole and split KV ranges, with and without staged page
ids, against the oracle; the plain plan gives the same rows within the
output's rounding."""
import math

import numpy as np
import pytest
import torch

from kunserve_amd import PrefillPlan, _lib, paged_prefill
from oracle import paged_attention_ref as ref

from helpers import (ATOL, ATOL_BF16, compact_for_oracle, max_abs, random_pool, random_tensor,
                     table_from_csr, to_numpy)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("ratio,hkv", [(2, 2), (3, 2), (5, 1), (7, 2), (8, 1), (16, 1)])
@pytest.mark.parametrize("num_cus", [1, 256])
def test_packed_rows_match_the_oracle(device, ratio, hkv, head_dim, num_cus, dtype):
    rng = np.random.default_rng(ratio + head_dim)
    tile = (128 if head_dim == 256 else 256) // ratio     # tokens per tile
    q_lens = np.array([1, tile, tile + 1, max(1, tile - 1), 70, 2 * tile + 3], dtype=np.int32)
    kv = (q_lens + np.array([300, 0, 63, 64, 1000, 129])).astype(np.int32)
    need = (kv + 15) // 16
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    npg = int(indptr[-1]) + 3
    indices = rng.permutation(npg)[:indptr[-1]].astype(np.int32)
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    hq = ratio * hkv
    pool = random_pool(npg, 1, hkv, 16, head_dim, device, 5, dtype=dtype)
    q = random_tensor((int(qi[-1]), hq, head_dim), device, 6, dtype=dtype)
    plan = PrefillPlan(qi, kv, hq, hkv, device, num_cus=num_cus, head_dim=head_dim)
    records = plan.plan_host[:6 * plan.info.num_tiles].reshape(-1, 6)
    assert np.all(records[records[:, 0] >= 0][:, 2] < 0)
    assert (plan.info.num_merge > 0) == (num_cus == 256)
    table = table_from_csr(indptr, indices, kv, device)
    qid = torch.from_numpy(qi).to(device)
    out = paged_prefill(pool, 0, table, qid, q, plan)
    torch.cuda.synchronize()
    k, v, ip, ix = compact_for_oracle(pool, 0, indptr, indices)
    want = ref.prefill_attention(to_numpy(q), qi, k, v, 0, ip, ix, kv, 1 / math.sqrt(head_dim))
    tol = ATOL_BF16 if dtype == torch.bfloat16 else ATOL
    assert max_abs(out, want) <= tol
    # rows too long for the staged page ids: the same results, bit for bit
    plan.info.max_kv_len = 1 << 20
    again = paged_prefill(pool, 0, table, qid, q, plan)
    torch.cuda.synchronize()
    assert torch.equal(again, out)
