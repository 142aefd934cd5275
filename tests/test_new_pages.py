"""kunserve_new_pages_private on random tables, and its cost: the step's, not
the pool's."""
import time

import numpy as np

from kunserve_amd import _lib


def _private(tables, q, kv, ps, num_pages):
    indptr = np.concatenate([[0], np.cumsum([len(t) for t in tables])]).astype(np.int32)
    indices = np.array([p for t in tables for p in t], dtype=np.int32)
    qi = np.concatenate([[0], np.cumsum(q)]).astype(np.int32)
    lens = np.array(kv, dtype=np.int32)
    return _lib.call("kunserve_new_pages_private", indptr.ctypes.data, indices.ctypes.data,
                     qi.ctypes.data, lens.ctypes.data, len(tables), ps, num_pages)


def test_agrees_with_a_count_of_the_pages():
    rng = np.random.default_rng(0)
    said = [0, 0]
    for _ in range(1500):
        rows, ps = int(rng.integers(0, 9)), int(rng.choice([4, 16]))
        q = rng.integers(0, 3 * ps, rows).tolist()
        kv = [int(n + rng.integers(0, 4 * ps)) for n in q]
        need = [-(-n // ps) for n in kv]
        pages = 4 + 3 * sum(need)
        ids = rng.permutation(pages)[:sum(need)].tolist()
        if ids and rng.integers(2):     # one page twice, or one outside the pool
            ids[int(rng.integers(len(ids)))] = int(rng.choice([ids[0], ids[-1], -1, pages]))
        tables = [[ids.pop() for _ in range(n)] for n in need]
        everywhere = [p for t in tables for p in t]
        new = [p for t, n, m in zip(tables, q, kv) if n for p in t[(m - n) // ps:(m - 1) // ps + 1]]
        want = int(all(0 <= p < pages and everywhere.count(p) == 1 for p in new))
        assert _private(tables, q, kv, ps, pages) == want, (tables, q, kv, ps)
        said[want] += 1
    assert min(said) > 100


def test_cost_does_not_grow_with_the_pool():
    """A byte of each page cleared per call would take a second for a few calls."""
    tables = [[5, 2**31 - 2], [7]]
    t = time.perf_counter()
    for _ in range(20):
        assert _private(tables, [1, 1], [20, 3], 16, 2**31 - 1) == 1
    assert time.perf_counter() - t < 1.0
