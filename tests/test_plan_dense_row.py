"""The MFMA plan of patterns with rows far wider than the rest, on the host: the
plain greedy colouring at hundreds to thousands of colours, and time and memory
that grow with a dense row as its pairs do, not with its cube."""
import resource
import time

import numpy as np
import pytest

from rsatb_amd import _lib
from test_plan_wide import plain_order


def hub_pattern(n):
    """Row 0 holds every column, the others column 0 and their own."""
    rows = [np.arange(n)] + [np.array([0, i]) for i in range(1, n)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    return rp, np.concatenate(rows).astype(np.int32)


@pytest.mark.parametrize("widest", [511, 512, 513, 600, 1100])
def test_more_colours_than_words(widest):
    n = 1200
    rng = np.random.default_rng(widest)
    rows = [rng.integers(0, n, rng.integers(0, 4)) for _ in range(n)]
    rows[n // 2] = rng.permutation(n)[:widest]
    rows[n // 3] = rng.permutation(n)[:widest - 7]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    ci = np.concatenate(rows).astype(np.int32)
    sched, kperm, _ = _lib.mfma_plan(rp, ci)
    assert np.array_equal(kperm, plain_order_fast(rp, ci, sched))


def plain_order_fast(rp, ci, sched):
    # plain_order with the columns near a column as an array
    n = len(rp) - 1
    row_of = np.repeat(np.arange(n), np.diff(rp))
    by_col = np.argsort(ci, kind="stable")
    cp = np.concatenate([[0], np.cumsum(np.bincount(ci, minlength=n))])
    col = np.full(n, -1)
    for r in sched:
        for c in ci[rp[r]:rp[r + 1]]:
            if col[c] >= 0:
                continue
            near = [col[ci[rp[q]:rp[q + 1]]] for q in row_of[by_col[cp[c]:cp[c + 1]]]]
            taken = np.zeros(n + 1, bool)
            taken[np.concatenate(near)] = True  # the entry of -1 is the last, never free's answer below n
            col[c] = int(np.argmin(taken[:n]))
    return np.concatenate([sorted(range(rp[r], rp[r + 1]), key=lambda p: (col[ci[p]], ci[p], p)) for r in range(n)])


def test_the_fast_reference_is_the_plain_one():
    rng = np.random.default_rng(0)
    rows = [rng.integers(0, 90, rng.integers(0, 5)) for _ in range(90)]
    rows[4] = rng.permutation(90)[:80]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    ci = np.concatenate(rows).astype(np.int32)
    sched, _, _ = _lib.mfma_plan(rp, ci)
    assert np.array_equal(plain_order_fast(rp, ci, sched), plain_order(rp, ci, sched))


def test_a_dense_row_costs_its_pairs():
    """Doubling the row quadruples the walks (a factor of 4; its cube would be
    8) and takes memory in proportion: at most 1 KB a row of the pattern."""
    def cost(n):
        rp, ci = hub_pattern(n)
        t = time.process_time()
        _lib.mfma_plan(rp, ci)
        return time.process_time() - t

    cost(1000)
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    small = min(cost(8000) for _ in range(3))
    large = min(cost(32000) for _ in range(2))
    assert large < 32 * small  # 16 by pairs, 64 by the cube
    assert resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before < 32000
