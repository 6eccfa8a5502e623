"""The block order of the MFMA plan against the plain greedy colouring it
states, on the host: rows with more columns than one word of colours holds (65
and 130 colours), unsorted rows and repeated columns, empty rows."""
import numpy as np
import pytest

from rsatb_amd import _lib


def plain_order(rp, ci, sched):
    # the smallest colour that no column sharing a row with c holds, columns in
    # the order they first appear in the schedule
    n = len(rp) - 1
    rows_of = [[] for _ in range(n)]
    for r in range(n):
        for c in ci[rp[r]:rp[r + 1]]:
            rows_of[c].append(r)
    col = [-1] * n
    for r in sched:
        for c in ci[rp[r]:rp[r + 1]]:
            if col[c] >= 0:
                continue
            near = {col[x] for q in rows_of[c] for x in ci[rp[q]:rp[q + 1]]}
            col[c] = next(k for k in range(n) if k not in near)
    return np.concatenate([sorted(range(rp[r], rp[r + 1]), key=lambda p: (col[ci[p]], ci[p], p)) for r in range(n)])


@pytest.mark.parametrize("n,widest,seed", [(40, 5, 1), (200, 65, 2), (300, 130, 3), (64, 64, 4)])
def test_block_order_is_the_greedy_colouring(n, widest, seed):
    rng = np.random.default_rng(seed)
    rows = [rng.integers(0, n, rng.integers(0, 6)) for _ in range(n)]  # unsorted, with repeats, some empty
    rows[n // 2] = rng.permutation(n)[:widest]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    ci = np.concatenate(rows).astype(np.int32)
    sched, kperm, _ = _lib.mfma_plan(rp, ci)
    assert sorted(sched) == list(range(n))
    assert np.array_equal(kperm, plain_order(rp, ci, sched))
