"""A step whose output buffer is also an input. Launches that append read the
step's k and v while they write out, so with out in k's or v's memory the
append is a launch of its own and the result that of a separate buffer."""
import ctypes

import numpy as np
import pytest
import torch

from kunserve_amd import AttentionStep, _lib

from helpers import random_pool, random_tensor


def _overlap(a, heads_a, b, heads_b, tokens, dim):
    ta, tb = _lib.Tensor3(*a), _lib.Tensor3(*b)
    return _lib.call("kunserve_tensors_overlap", ctypes.byref(ta), heads_a, ctypes.byref(tb),
                     heads_b, tokens, dim)


def _elements(t, heads, tokens, dim):
    base, ts, hs = t
    i = np.arange(tokens)[:, None, None] * ts + np.arange(heads)[None, :, None] * hs
    return set((base + 2 * (i + np.arange(dim))).reshape(-1).tolist())


def test_tensors_overlap_never_misses_a_shared_element():
    rng = np.random.default_rng(0)
    exact = 0
    for _ in range(4000):
        tokens, dim = int(rng.integers(0, 5)), int(rng.choice([1, 4]))
        heads = rng.integers(0, 4, 2).tolist()
        strides = [[int(rng.integers(-20, 40)), int(rng.integers(-6, 9))] for _ in range(2)]
        if rng.integers(2):
            strides[1][0] = strides[0][0]
        a = (4096 + 2 * int(rng.integers(0, 60)), *strides[0])
        b = (4096 + 2 * int(rng.integers(0, 60)), *strides[1])
        shared = bool(_elements(a, heads[0], tokens, dim) & _elements(b, heads[1], tokens, dim))
        said = _overlap(a, heads[0], b, heads[1], tokens, dim)
        assert said or not shared, (a, b, heads, tokens, dim)
        exact += said == shared
    assert exact > 2000


@pytest.mark.parametrize("at,heads,overlaps", [
    (0, 8, 0), (8, 2, 1), (10, 2, 1), (7, 2, 1), (9, 1, 1), (0, 12, 1), (11, 8, 1), (12, 8, 0),
    (-8, 8, 1), (-1, 2, 1), (-12, 8, 0), (-5, 2, 1)])
def test_slices_of_one_projection_are_apart(at, heads, overlaps):
    """Rows of 12 heads: k at heads 8 and 9, v at 10 and 11; out `heads` heads
    from head `at` on (of this row, a later or an earlier one)."""
    d, base = 64, 1 << 20
    out = (base + 2 * d * at, 12 * d, d)
    said = [_overlap(out, heads, (base + 2 * d * h, 12 * d, d), 2, 5, d) for h in (8, 10)]
    assert max(said) == overlaps


def _tables(kv, ps, seed):
    need = [-(-n // ps) for n in kv]
    perm = np.random.default_rng(seed).permutation(sum(need) + 2).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n])
        at += n
    return tables, sum(need) + 2


@pytest.mark.gpu
@pytest.mark.parametrize("into", ["k", "v"])
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(8, 8), (8, 2)])
def test_step_writes_its_output_over_an_input(device, into, hd, hq, hkv):
    """Chunks of several q tiles beside decode rows. With GQA, out covers k or v
    and the heads before it in one projection."""
    rows = [(700, 0, 0), (513, 100, 0), (1, 900, 1), (65, 31, 0), (1, 40, 1), (2, 15, 0)]
    q_lens = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    tables, npg = _tables(kv, 16, hd)
    first = [n if d else n - t for (t, _, d), n in zip(rows, kv)]
    pools = [random_pool(npg, 1, hkv, 16, hd, device, 3) for _ in range(2)]
    steps = [AttentionStep(p, hq, q_lens, first, [1 - r[2] for r in rows], tables) for p in pools]
    assert steps[0]._step.appends == 1
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, 2.0)
    proj = random_tensor((T, hq + 2 * hkv, hd), device, 5)
    at = {"k": hq, "v": hq + hkv}
    k, v = (proj[:, at[n]:at[n] + hkv] for n in "kv")
    want = steps[0].run(0, q, k.clone(), v.clone())
    end = at[into] + hkv
    out = proj[:, end - hq:end]
    got = steps[1].run(0, q, k, v, out=out)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert torch.equal(pools[0].k, pools[1].k) and torch.equal(pools[0].v, pools[1].v)


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(8, 8), (8, 2)])
def test_step_writes_its_output_over_q(device, hd, hq, hkv):
    """Whole and split rows: every reader of a q row has read it before its out
    is written."""
    rows = [(300, 0, 0), (31, 1200, 0), (1, 900, 1), (65, 31, 0), (1, 40, 1)]
    q_lens = [r[0] for r in rows]
    kv = [r[0] + r[1] for r in rows]
    tables, npg = _tables(kv, 16, hd)
    first = [n if d else n - t for (t, _, d), n in zip(rows, kv)]
    pool = random_pool(npg, 1, hkv, 16, hd, device, 3)
    step = AttentionStep(pool, hq, q_lens, first, [1 - r[2] for r in rows], tables)
    assert step.prefill.plan.info.num_merge > 0 and step.decode.plan.info.num_merge > 0
    T = sum(q_lens)
    q = random_tensor((T, hq, hd), device, 4, 2.0)
    k, v = (random_tensor((T, hkv, hd), device, s) for s in (5, 6))
    want = step.run(0, q, k, v).clone()
    got = step.run(0, q, k, v, out=q)
    torch.cuda.synchronize()
    assert got is q and torch.equal(got, want)


@pytest.mark.gpu
def test_step_of_no_rows(device):
    pool = random_pool(4, 1, 2, 16, 128, device, 3)
    step = AttentionStep(pool, 4, [], [], [], [])
    q = torch.empty((0, 4, 128), dtype=torch.float16, device=device)
    k = torch.empty((0, 2, 128), dtype=torch.float16, device=device)
    assert step.run(0, q, k, k.clone()).shape == q.shape
