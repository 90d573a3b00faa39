"""Run directory of B over more than one range of 512 blocks, where each
row's entries in a range are searched: rows and columns around the ranges' and
row groups' edges, empty rows, rows that skip ranges, against the oracle on
columns relabelled in order -- and the time to make it, which follows B's
entries and not its columns."""
from __future__ import annotations

import time

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

RANGE = 512 * 1024


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate(lists).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


def _handle():
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    h.set_tuning({"row_bins": (0, 0, 0)})        # every row a big row
    h.set_item_order(0)                          # in column order
    return h


@pytest.mark.parametrize("n", [1, 33, 255, 256, 257, 600])
@pytest.mark.parametrize("k", [RANGE, RANGE + 1, 2 * RANGE, 2 * RANGE + 1, 4 * RANGE + 77, 2**26 + 5, 2**31 - 1])
def test_ranges_of_blocks(n, k):
    rng = np.random.default_rng(n + k % 1000)
    edges = np.unique([c for b in range(0, min(k // RANGE, 9) + 1) for d in (-1025, -1, 0, 1, 1024)
                       if 0 <= (c := b * RANGE + d) < k] + [k - 1])
    brows = []
    for t in range(n):
        kind = t % 6
        if kind == 0:
            c = rng.choice(edges, 5)
        elif kind == 1:
            c = np.array([], dtype=np.int64)
        elif kind == 2:
            c = edges
        elif kind == 3:
            c = rng.integers(0, k, 300)
        elif kind == 4:
            c = min(k - 1, RANGE) - 40 + np.arange(80)
        else:
            c = rng.integers(k - k // 3, k, 50)
        brows.append(np.unique(c[c < k]))
    arows = [np.arange(n), np.arange(0, n, 3), np.array([n - 1]), np.unique(rng.integers(0, n, 90))]
    A, B = _csr(arows, rng), _csr(brows, rng)
    used, at = np.unique(B[1], return_inverse=True)
    ic, jc, c = O.csr_spgemm(len(arows), used.size, A, (B[0], at.astype(np.int32), B[2]))
    want = (ic, used[jc].astype(np.int32), c)
    h = _handle()
    h.set_block_pointer_budget(6 << 30)
    dA = tsg.DeviceCsr.from_host(len(arows), n, *A)
    dB = tsg.DeviceCsr.from_host(n, k, *B)
    for bitmap in (-1, 0):
        h.set_bitmap_budget(bitmap)
        assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()


def test_time_to_make_it_follows_the_entries():
    """512 rows of 4000 entries over 2^28 columns: the symbolic phase takes less
    than 4 times as long with the directory as without (17 times when every
    range read every entry)."""
    import torch
    rng = np.random.default_rng(0)
    n, per, k = 512, 4000, 2**28
    col = np.sort(rng.integers(0, k, (n, per)), axis=1)
    B = tsg.DeviceCsr.from_host(n, k, np.arange(0, n * per + 1, per), col.ravel(), np.ones(n * per))
    A = tsg.DeviceCsr.from_host(16, n, np.arange(0, 16 * 32 + 1, 32),
                                np.sort(rng.integers(0, n, (16, 32)), axis=1).ravel(), np.ones(512))
    h = _handle()
    took = []
    for budget in (6 << 30, 0):                  # the directory, and searches in B's rows
        h.set_block_pointer_budget(budget)
        best = 1e9
        for _ in range(4):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            h.symbolic(A, B)
            best = min(best, time.perf_counter() - t0)
        took.append(best)
    h.close()
    assert took[0] < 4 * took[1], took
