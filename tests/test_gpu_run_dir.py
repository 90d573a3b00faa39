"""Big rows in column order, B cut by its run directory: B rows and columns
around the directory's groups of 32 rows and blocks of 1024 columns, spans that
start inside a band, coarse blocks and no directory, against the oracle."""
from __future__ import annotations

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


def _check(m, n, k, A, B, fp, budgets):
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    h.set_tuning({"row_bins": (0, 0, 0)})        # every row a big row
    h.set_item_order(0)                          # in column order
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for budget in budgets:
        for bitmap in (-1, 0):                   # rank tables, hash tables
            h.set_block_pointer_budget(budget)
            h.set_bitmap_budget(bitmap)
            assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 300, 1000])
@pytest.mark.parametrize("k", [1, 1023, 1025, 65536, 65537, 200_003])
def test_rows_and_columns_at_the_edges(n, k, fp):
    """B's rows: empty ones, single entries at block edges, runs over edges,
    random ones, repeated columns.  The budgets give the finest blocks, coarser
    ones (where the whole directory takes more) and none."""
    rng = np.random.default_rng(n + k)
    edges = np.array([c for b in (0, 1024, 8192, 65536, 131072, k) for c in (b - 1, b, b + 1)
                      if 0 <= c < k])
    brows = []
    for t in range(n):
        kind = t % 6
        if kind == 0:
            c = rng.choice(edges, 2)
        elif kind == 1:
            c = np.array([], dtype=np.int64)
        elif kind == 2:
            lo = int(rng.choice(edges))
            c = np.arange(lo, min(k, lo + 70))
        elif kind == 3:
            c = rng.integers(0, k, 90)
        elif kind == 4:
            c = np.unique(rng.integers(k // 2, k, 400))
        else:
            c = rng.integers(k - k // 5 - 1, k, 30)
        brows.append(np.sort(c))
    arows = [np.arange(n), np.arange(0, n, 3), np.array([n - 1]), np.arange(4, n, 6),
             rng.integers(0, n, 200)]
    A, B = _csr(arows, rng), _csr(brows, rng)
    fine = 2 * ((k + 65535) // 65536) * 64 * ((n + 31) // 32) * 12
    _check(len(arows), n, k, A, B, fp, (-1, fine // 2 + 8 * B[1].size, 0))


@pytest.mark.parametrize("cols", [1, 200, 511, 512])
def test_a_single_wide_item(cols):
    """One row whose outputs make one item of up to a whole band."""
    rng = np.random.default_rng(cols)
    k = 3 * 65536
    c = 65536 + np.sort(rng.choice(65536, cols, replace=False))
    A, B = _csr([np.array([0, 1])], rng), _csr([c, c], rng)
    _check(1, 2, k, A, B, tsg.FP_FUSED, (-1, 0))
