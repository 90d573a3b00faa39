"""Rows of 1024 to 1536 products around the limits of their kernel: products,
A entries, outputs summed at a time; spread and repeated columns."""
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


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("k", [400, 1500, 40_000, 3_000_000])
@pytest.mark.parametrize("repeat", [False, True])
def test_rows_at_the_limits(k, repeat, fp):
    """One row per number of products and A entries; its B rows are random (of
    k columns) and, with repeat, name columns twice."""
    rng = np.random.default_rng(k)
    arows, brows = [], []
    for prod in (1024, 1025, 1088, 1152, 1153, 1300, 1535, 1536, 1537):
        for ent in (4, 16, 63, 64, 65):
            cuts = np.sort(rng.choice(np.arange(1, prod), ent - 1, replace=False))
            sizes = np.minimum(np.diff(np.concatenate([[0], cuts, [prod]])), k)
            row = []
            for n in sizes:
                c = rng.integers(0, k, n) if repeat else rng.choice(k, n, replace=False)
                row.append(len(brows))
                brows.append(np.sort(c))
            arows.append(row)

    A, B = _csr(arows, rng), _csr(brows, rng)
    m, n = len(arows), len(brows)
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for bins in ((64, 256, 1024), (64, 256, 512)):     # with these rows' kernel, without
        h.set_tuning({"row_bins": bins})
        assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()


@pytest.mark.parametrize("big", [1, 3, 40])
def test_few_big_rows_of_a_large_b(big):
    """Big rows of 3000 products each, fewer and more than a quarter of B's
    entries together: only the B rows they name are packed, or all."""
    rng = np.random.default_rng(big)
    n = k = 3000
    brows = [np.sort(rng.choice(k, 50, replace=False)) for _ in range(n)]
    arows = [np.sort(rng.choice(n, 60 if i < big else 2, replace=False)) for i in range(200)]
    A, B = _csr(arows, rng), _csr(brows, rng)
    want = O.csr_spgemm(len(arows), k, A, B, fused=True)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=tsg.FP_FUSED)
    dA, dB = tsg.DeviceCsr.from_host(len(arows), n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for order in (1 << 18, 0):                   # rows' order, column order
        h.set_item_order(order)
        assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()
