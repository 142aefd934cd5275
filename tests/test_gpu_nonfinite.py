"""Infinite and NaN values in V stay in their dim: decode outputs are infinite
or NaN exactly where the oracle's are and finite, with the oracle's values,
everywhere else, whatever the partition, the wave and the lane that meet them,
and whichever launch combines the partitions; split prefill rows that see no
key of a split take nothing from it."""
import math

import numpy as np
import pytest
import torch

from kunserve_amd import AttentionStep, DecodePlan, paged_decode
from oracle import paged_attention_ref as ref

from helpers import (ATOL, ATOL_BF16, compact_for_oracle, random_pool, random_tensor,
                     table_from_csr, to_numpy)

KV = np.array([257, 1, 33, 100, 700, 2048, 64], dtype=np.int32)


def _check(got, want, tol):
    got = to_numpy(got).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert ok.any() and np.abs(got[ok] - want[ok]).max() <= tol


def _marked_rows(hkv, hd, dtype, device):
    """A pool, its table and lists, with values at the ends of rows, partitions
    of 256 and steps, two of one sign and both signs in one dim; row 6 has none."""
    need = (KV + 15) // 16
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    npg = int(indptr[-1]) + 1
    indices = np.random.default_rng(hd + hkv).permutation(npg)[:indptr[-1]].astype(np.int32)
    pool = random_pool(npg, 1, hkv, 16, hd, device, 5, dtype=dtype)
    inf, nan = math.inf, math.nan
    for b, t, h, d, x in [
            (0, 256, 0, 3, inf), (0, 0, hkv - 1, hd - 1, -inf), (1, 0, 0, hd // 2 + 5, nan),
            (2, 32, 0, 0, inf), (2, 1, 0, 0, inf), (2, 7, 0, 1, inf), (2, 8, 0, 1, -inf),
            (3, 63, hkv - 1, 17, -inf), (3, 64, hkv - 1, 18, inf), (4, 699, 0, 9, inf),
            (4, 300, 0, 10, nan), (5, 2047, 0, 40, inf), (5, 5, hkv - 1, hd - 2, -inf),
            (5, 1100, 0, 41, -inf)]:
        pool.v[int(indices[indptr[b] + t // 16]), 0, h, t % 16, d] = x
    return pool, indptr, indices


def _oracle(pool, indptr, indices, q):
    k, v, ip, ix = compact_for_oracle(pool, 0, indptr, indices)
    return ref.decode_attention(to_numpy(q), k, v, 0, ip, ix, KV, 1 / math.sqrt(pool.head_dim))


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (4, 2), (6, 2), (8, 2), (8, 1), (12, 1), (32, 1)])
def test_decode_keeps_nonfinite_values_in_their_dim(device, hq, hkv, hd, dtype):
    pool, indptr, indices = _marked_rows(hkv, hd, dtype, device)
    q = random_tensor((len(KV), hq, hd), device, 6, 0.5, dtype=dtype)
    table = table_from_csr(indptr, indices, KV, device)
    want = _oracle(pool, indptr, indices, q)
    for part in (0, 256, 4096):
        got = paged_decode(pool, 0, table, q, DecodePlan(KV, hq, hkv, device, part))
        _check(got, want, ATOL if dtype == torch.float16 else ATOL_BF16)


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (4, 2), (6, 2), (8, 2), (32, 1)])
def test_decode_step_combines_nonfinite_partials(device, hq, hkv, hd, dtype):
    """A step's launch combines rows of 1 to 8 partitions, whose last tokens come
    from its k and v; the last partitions hold such values too."""
    pool, indptr, indices = _marked_rows(hkv, hd, dtype, device)
    q = random_tensor((len(KV), hq, hd), device, 6, 0.5, dtype=dtype)
    want = _oracle(pool, indptr, indices, q)
    last = [(int(indices[indptr[b] + (n - 1) // 16]), (n - 1) % 16) for b, n in enumerate(KV)]
    k, v = (torch.stack([x[p, 0, :, t] for p, t in last]) for x in (pool.k, pool.v))
    tables = [indices[indptr[b]:indptr[b + 1]].tolist() for b in range(len(KV))]
    step = AttentionStep(pool, hq, [1] * len(KV), KV, [0] * len(KV), tables,
                         decode_part_tokens=256)
    assert step._step.appends == 1 and step._step.num_counters > 0
    _check(step.run(0, q, k, v), want, ATOL if dtype == torch.float16 else ATOL_BF16)


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("value", [math.inf, math.nan])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (4, 2)])
@pytest.mark.parametrize("mixed", [False, True])
def test_prefill_rows_before_a_split_take_nothing_from_it(device, hq, hkv, hd, value, mixed):
    """31 tokens on both sides of position 768, where the last of 4 splits
    begins, and a value that only tokens from 768 on see."""
    q_lens, prefix = [31, 31], [752, 752]
    kv = [783, 783]
    if mixed:
        q_lens, kv = q_lens + [1], kv + [300]
    need = [-(-n // 16) for n in kv]
    npg = sum(need)
    perm = np.random.default_rng(hd).permutation(npg).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    pool = random_pool(npg, 1, hkv, 16, hd, device, 3)
    step = AttentionStep(pool, hq, q_lens, prefix + kv[2:], [1, 1] + [0] * mixed, tables)
    info = step.prefill.plan.info
    assert info.kv_chunk == 256 and step._step.num_prefill_counters > 0
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, 0.5)
    k, v = (random_tensor((T, hkv, hd), device, s) for s in (5, 6))
    v[18, 0, hd - 3] = value     # position 770 of the first row
    kh, vh = to_numpy(pool.k), to_numpy(pool.v)
    out = step.run(0, q, k, v)
    indptr = np.concatenate([[0], np.cumsum(need)]).astype(np.int32)
    indices = np.array([p for t in tables for p in t], dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    lens = np.array(kv, dtype=np.int32)
    ref.append_kv(kh, vh, 0, indptr, indices, lens, qi, to_numpy(k), to_numpy(v))
    want = ref.prefill_attention(to_numpy(q), qi, kh, np.where(np.isfinite(vh), vh, 0), 0, indptr,
                                 indices, lens, 1 / math.sqrt(hd))
    _check(out[:16], want[:16], ATOL)
    _check(out[31:], want[31:], ATOL)
