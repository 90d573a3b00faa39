"""Big rows with few A entries and products against B's entries, for which
only the B rows they name are packed: numbers of A entries around the groups
that a block takes, rows of none, one and many entries in one group, long and
empty B rows, B rows named twice, against the oracle -- and the time with one
long row of A."""
from __future__ import annotations

import time

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate(lists).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("lens", [[1], [63], [64], [65], [1, 62, 1], [40, 40, 40], [64, 64],
                                  [1] * 70, [127, 1], [3, 1500, 2], [130, 0, 700],
                                  [1] * 100, [4000]])
@pytest.mark.parametrize("order", [0, 1 << 60])
def test_groups_of_entries(lens, order, fp):
    rng = np.random.default_rng(sum(lens) + len(lens))
    n, k = 6000, 70_001
    brows = [np.unique(rng.integers(0, k, int(x)))
             for x in rng.choice([0, 1, 2, 7, 30], n)]
    long = int(rng.integers(12, n))
    brows[long] = np.unique(rng.integers(0, k, 3000))
    for t in range(12):
        brows[t] = np.arange(t, k)                        # not named: the most of B
    arows = []
    for x in lens:
        row = 12 + rng.choice(n - 12, x, replace=False)
        if x:
            row[0] = long
        arows.append(np.sort(row))
    A, B = _csr(arows, rng), _csr(brows, rng)
    products = sum(len(brows[t]) for r in arows for t in r)
    named = products * 4 < B[1].size and sum(lens) * 256 < B[1].size
    assert named == (lens not in ([1] * 100, [4000]))     # these: all of B packed
    m = len(arows)
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    h.set_tuning({"row_bins": (0, 0, 0)})                 # every row a big row
    h.set_item_order(order)
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()


def test_time_with_a_long_row():
    """The numeric phase of a banded matrix with one row of 12,000 entries: less
    than 20 times that of the band alone (a wave for the row's packing: 45)."""
    import torch
    n, half, long = 1 << 19, 3, 12_000
    rng = np.random.default_rng(1)
    off = np.arange(-half, half + 1)
    took = []
    for extra in (0, long):
        key = (np.arange(n)[:, None] * n + np.clip(np.arange(n)[:, None] + off, 0, n - 1)).ravel()
        key = np.unique(np.concatenate([key, 777 * n + rng.integers(0, n, extra)]))
        ptr = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(key // n, minlength=n), out=ptr[1:])
        A = tsg.DeviceCsr.from_host(n, n, ptr, key % n, np.ones(key.size))
        h = tsg.Handle(0, method=tsg.METHOD_ROW)
        ic, nnz = h.symbolic(A, A)
        jc = torch.empty(nnz, dtype=torch.int32, device="cuda:0")
        c = torch.empty(nnz, dtype=torch.float64, device="cuda:0")
        best = 1e9
        for _ in range(5):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            h.numeric(A, A, ic, jc, c)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        took.append(best)
        h.close()
    assert took[1] < 20 * took[0], took
