"""Run directory of B with coarse blocks -- 2048 to 65536 columns, the rest by
search inside a run -- as a budget gives them: B rows and columns around block
edges, against the oracle, with the form that was built asked of the plan."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

CHUNK = 8192                                     # cells scanned together
LEVELS = 7


def _bytes(n, k, nnz, c):
    """The directory with finest blocks of 1024 << c columns."""
    nblk = -(-k // 65536) << (6 - c)
    levels = LEVELS - c
    cells = (2 * nblk - (2 * nblk >> levels)) * (-(-n // 32))
    return -(-cells // CHUNK) * (CHUNK * 12 + 8) + levels * nnz * 8


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate(lists).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("n,k", [(2000, 200_003), (700, 1_000_001), (1025, 65536 * 9)])
@pytest.mark.parametrize("repeat", [False, True])
def test_coarse_blocks(n, k, repeat, fp):
    rng = np.random.default_rng(n + k)
    edges = np.array([c for b in range(0, k + 65537, 2048) for c in (b - 1, b, b + 1)
                      if 0 <= c < k])
    brows = []
    for t in range(n):
        kind = t % 5
        if kind == 0:
            c = rng.choice(edges, 8)
        elif kind == 1:
            c = np.array([], dtype=np.int64)
        elif kind == 2:
            lo = int(rng.choice(edges))
            c = np.arange(lo, min(k, lo + 40))
        elif kind == 3:
            c = rng.integers(0, k, 30)
        else:
            lo = int(rng.integers(0, k - 5000))
            c = rng.integers(lo, lo + 5000, 60)
        c = np.unique(c)
        if repeat and c.size > 2:                # a column twice: rows not strict
            c[1] = c[0]
        brows.append(c)
    arows = [np.arange(n), np.arange(0, n, 3), np.array([n - 1]), np.arange(4, n, 5),
             np.unique(rng.integers(0, n, 150))]
    A, B = _csr(arows, rng), _csr(brows, rng)
    m, nnz = len(arows), B[1].size
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    h.set_tuning({"row_bins": (0, 0, 0)})        # every row a big row
    h.set_item_order(0)                          # in column order
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    built = []
    for c in (0, 1, 3, 5, 6, 7):                 # 7: not even the coarsest
        h.set_block_pointer_budget(_bytes(n, k, nnz, min(c, 6)) - (c == 7))
        for bitmap in (-1, 0):                   # rank tables, hash tables
            h.set_bitmap_budget(bitmap)
            assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
            built.append(tsg.load().tsg_plan_dir_shift(h._h))
    h.close()
    assert built == [x for c in (10, 11, 13, 15, 16, 0) for x in (c, c)]
