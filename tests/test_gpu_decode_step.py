"""Decode-only steps in one launch per layer: the decode kernel appends the
rows' new K/V and its last workgroup per split row combines the partials.
The pages hold the appended bytes, the outputs match the oracle on the pages
after the append, repeated layers and graph replays agree bit for bit (the
counters come back to zero), and a step whose rows share a last page appends
in a launch of its own."""
import math

import numpy as np
import pytest
import torch

from kunserve_amd import AttentionStep, _lib
from oracle import paged_attention_ref as ref

from helpers import ATOL, ATOL_BF16, max_abs, random_pool, random_tensor, to_numpy


@pytest.mark.parametrize("rows,q,kv,private", [
    ([[0, 1], [2]], [1, 1], [20, 3], 1), ([[0, 1], [1]], [1, 1], [20, 3], 0),
    ([[0, 1], [0, 2]], [1, 1], [20, 20], 1), ([[3, 4], [4, 2]], [1, 1], [17, 17], 0),
    ([[5, 5]], [1], [17], 0), ([], [], [], 1), ([[], [1]], [0, 1], [0, 1], 1),
    ([[0, 1, 2], [0, 3]], [16, 1], [48, 32], 1),     # a shared prefix page
    ([[0, 1, 2], [1, 3]], [16, 1], [48, 32], 1),
    ([[0, 1, 2], [1, 3]], [17, 1], [48, 32], 0),     # page 1 holds row 0's first new token
    ([[0, 1, 2], [2, 3]], [40, 2], [48, 32], 0)])
def test_new_pages_private(rows, q, kv, private):
    indptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    indices = np.array([p for r in rows for p in r], dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q)]).astype(np.int32)
    lens = np.array(kv, dtype=np.int32)
    assert _lib.call("kunserve_new_pages_private", indptr.ctypes.data, indices.ctypes.data,
                     qi.ctypes.data, lens.ctypes.data, len(rows), 16, 8) == private


def _step(kv, hq, hkv, hd, ps, dtype, device, part, shared_last=False):
    rng = np.random.default_rng(hq + hd)
    need = [-(-n // ps) for n in kv]
    npg = sum(need) + 4
    perm = rng.permutation(npg).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    if shared_last:
        tables[1][0] = tables[0][-1]
    pool = random_pool(npg, 2, hkv, ps, hd, device, 3, dtype=dtype)
    step = AttentionStep(pool, hq, [1] * len(kv), kv, [0] * len(kv), tables,
                         decode_part_tokens=part)
    n = len(kv)
    q = random_tensor((n, hq, hd), device, 4, 2.0, dtype=dtype)
    k = random_tensor((n, hkv, hd), device, 5, dtype=dtype)
    v = random_tensor((n, hkv, hd), device, 6, dtype=dtype)
    return pool, step, tables, q, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (4, 2), (8, 2), (6, 2), (32, 1)])
@pytest.mark.parametrize("shared_last", [False, True])
@pytest.mark.parametrize("longest", [2047, 2305])
def test_decode_step_appends_and_combines(device, hq, hkv, hd, dtype, shared_last, longest):
    """Rows whose new token is a partition's only one (257, 513), a page's
    first and last, a row of one token, and rows of 1 to 8 partitions, which
    the launch combines, or with one of 10 a merge launch. With a shared last page, row 1 (2 tokens)
    reads the token that row 0 appends to it."""
    kv = [257, 2 if shared_last else 1, 16, 17, 513, 256, longest, 2048, 100]
    pool, step, tables, q, k, v = _step(kv, hq, hkv, hd, 16, dtype, device, 256, shared_last)
    assert step._step.appends == (0 if shared_last else 1)
    assert step.decode.plan.info.num_merge == 4
    kh, vh = to_numpy(pool.k), to_numpy(pool.v)
    outs = [step.run(1, q, k, v) for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert (step._step.num_counters > 0) == (longest == 2047)
    assert step.counters is None or not step.counters.any().item()
    indptr = np.concatenate([[0], np.cumsum([len(t) for t in tables])]).astype(np.int32)
    indices = np.array([p for t in tables for p in t], dtype=np.int32)
    lens = np.array(kv, dtype=np.int32)
    ref.append_kv(kh, vh, 1, indptr, indices, lens, np.arange(len(kv) + 1, dtype=np.int32),
                  to_numpy(k), to_numpy(v))
    assert np.array_equal(to_numpy(pool.k), kh) and np.array_equal(to_numpy(pool.v), vh)
    want = ref.decode_attention(to_numpy(q), kh, vh, 1, indptr, indices, lens, 1 / math.sqrt(hd))
    assert max_abs(outs[0], want) <= (ATOL if dtype == torch.float16 else ATOL_BF16)


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 2)])
def test_decode_step_replays_in_a_graph(device, hq, hkv):
    kv = [700, 33, 2100]
    pool, step, _, q, k, v = _step(kv, hq, hkv, 128, 16, torch.float16, device, 256)
    out = torch.empty_like(q)
    want = [step.run(layer, q, k, v).clone() for layer in (0, 1)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    outs = [torch.empty_like(q) for _ in range(2)]
    with torch.cuda.graph(graph):
        for layer in (0, 1):
            step.run(layer, q, k, v, out=outs[layer])
    for _ in range(4):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want[0]) and torch.equal(outs[1], want[1])
        assert torch.equal(step.run(1, q, k, v, out=out), want[1])
        torch.cuda.synchronize()
