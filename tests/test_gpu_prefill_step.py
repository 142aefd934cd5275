"""Steps with split prefill rows, alone and beside split decode rows: the
prefill launch combines its splits itself, each row block by the last of its
waves to finish. Outputs match the oracle, and those of the two-launch path
within the output's rounding; repeated layers and graph replays agree bit
for bit and leave the counters zeroed."""
import math

import numpy as np
import pytest
import torch

from kunserve_amd import AttentionStep, paged_prefill
from oracle import paged_attention_ref as ref

from helpers import ATOL, ATOL_BF16, max_abs, random_pool, random_tensor, to_numpy


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 2), (6, 2)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("splits", [4, 5])
def test_prefill_step_combines_its_splits(device, hq, hkv, hd, dtype, mixed, splits):
    """Rows whose last tile holds 1, 31, 33 and all rows, of 1 to 4 splits, one
    whose last split holds keys that some of its rows do not see; with a longer
    prefix (5 and more splits) the merge is a launch of its own."""
    rows = [(1, 1023 if splits == 4 else 1600, 0), (31, 702, 0), (130, 401, 0), (257, 0, 0)]
    if mixed:
        rows = [(1, 2999, 1), rows[0], rows[1], (1, 40, 1), rows[2], rows[3]]
    q_lens = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    dec = [r[2] for r in rows]
    rng = np.random.default_rng(hq + hd)
    need = [-(-n // 16) for n in kv]
    npg = sum(need) + 4
    perm = rng.permutation(npg).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    pool = random_pool(npg, 1, hkv, 16, hd, device, 3, dtype=dtype)
    first = [n if d else n - t for t, n, d in zip(q_lens, kv, dec)]
    step = AttentionStep(pool, hq, q_lens, first, [1 - d for d in dec], tables)
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, 2.0, dtype=dtype)
    k = random_tensor((T, hkv, hd), device, 5, dtype=dtype)
    v = random_tensor((T, hkv, hd), device, 6, dtype=dtype)
    info = step.prefill.plan.info
    assert info.num_merge > 0 and info.kv_chunk == 256
    assert step._step.num_prefill_counters == (info.num_slots * info.tile_q // 32
                                               if splits == 4 else 0)
    assert (step.decode is not None) == mixed and step._step.appends == 1
    kh, vh = to_numpy(pool.k), to_numpy(pool.v)
    outs = [step.run(0, q, k, v).clone() for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert step.counters is None or not step.counters.any().item()
    tol = ATOL if dtype == torch.float16 else ATOL_BF16
    p = step.prefill
    two = outs[0].clone()
    paged_prefill(pool, 0, p.table, p.q_indptr, q, p.plan, out=two, q_start=p.tokens)
    torch.cuda.synchronize()
    assert max_abs(two, outs[0].float()) <= tol
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    indices = np.array([x for t in tables for x in t], dtype=np.int32)
    lens = np.array(kv, dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    ref.append_kv(kh, vh, 0, indptr, indices, lens, qi, to_numpy(k), to_numpy(v))
    assert np.array_equal(to_numpy(pool.k), kh) and np.array_equal(to_numpy(pool.v), vh)
    want = ref.prefill_attention(to_numpy(q), qi, to_numpy(pool.k), to_numpy(pool.v), 0, indptr,
                                 indices, lens, 1 / math.sqrt(hd))
    assert max_abs(outs[0], want) <= tol
    graph = torch.cuda.CUDAGraph()
    out = torch.empty_like(q)
    with torch.cuda.graph(graph):
        step.run(0, q, k, v, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])
        assert torch.equal(step.run(0, q, k, v), outs[0])
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 2), (10, 2), (7, 1)])
@pytest.mark.parametrize("ps", [4, 16, 256])
@pytest.mark.parametrize("shared", [False, True])
def test_prefill_step_appends_its_rows(device, monkeypatch, hq, hkv, hd, dtype, ps, shared):
    """Whole KV ranges: prefixes that end anywhere in a group of 4 tokens, in a
    page and in a KV tile, rows of several q tiles, packed rows whose tile ends
    inside a token, and a decode row. With `shared`, the decode row's table
    holds a page of another row's new tokens, and the append is a launch of
    its own."""
    from kunserve_amd import paged_kv
    monkeypatch.setattr(paged_kv, "_num_cus", lambda d: 1)
    rows = [(1, 63, 0), (2, 61, 0), (64, 0, 0), (1, 333, 1), (65, 5, 0), (130, 127, 0),
            (300, 258, 0), (3, 1, 0)]
    q_lens = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    dec = [r[2] for r in rows]
    rng = np.random.default_rng(hq + hd + ps)
    need = [-(-n // ps) for n in kv]
    npg = sum(need) + 4
    perm = rng.permutation(npg).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    if shared:
        tables[3][0] = tables[5][-1]
    pool = random_pool(npg, 2, hkv, ps, hd, device, 3, dtype=dtype)
    first = [n if d else n - t for t, n, d in zip(q_lens, kv, dec)]
    step = AttentionStep(pool, hq, q_lens, first, [1 - d for d in dec], tables)
    assert step.prefill.plan.info.num_merge == 0 and step._step.appends == (0 if shared else 1)
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, 2.0, dtype=dtype)
    # strided k and v, as slices of one projection
    kvt = random_tensor((T, 2 * hkv, hd), device, 5, dtype=dtype)
    k, v = kvt[:, :hkv], kvt[:, hkv:]
    kh, vh = to_numpy(pool.k), to_numpy(pool.v)
    out = step.run(1, q, k, v)
    again = step.run(1, q, k, v)
    torch.cuda.synchronize()
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    indices = np.array([x for t in tables for x in t], dtype=np.int32)
    lens = np.array(kv, dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    ref.append_kv(kh, vh, 1, indptr, indices, lens, qi, to_numpy(k), to_numpy(v))
    assert np.array_equal(to_numpy(pool.k), kh) and np.array_equal(to_numpy(pool.v), vh)
    assert torch.equal(out, again)
    want = ref.prefill_attention(to_numpy(q), qi, kh, vh, 1, indptr, indices, lens,
                                 1 / math.sqrt(hd))
    assert max_abs(out, want) <= (ATOL if dtype == torch.float16 else ATOL_BF16)
