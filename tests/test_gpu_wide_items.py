"""Big rows in column order: sparse stretches of a row run as wide items.  Rows
whose bands hold outputs around the items' limits, spread over the band or in
one window of it, against the oracle in both FP modes."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

BAND, WINDOW = 65536, 8192


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("spread", ["band", "window", "ends"])
@pytest.mark.parametrize("parts", [2, 9, 40])
def test_wide_items_at_their_limits(parts, spread, fp):
    """C's row has n distinct columns in each of three bands; the row's A
    entries name parts B rows that each hold a random half of them (and one
    that holds all), so every output sums several products."""
    rng = np.random.default_rng(parts)
    k = 3 * BAND + 517
    arows, brows = [], []
    for n in (1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1024, 1500):
        cols = []
        for band in range(3):
            lo, hi = band * BAND, min(k, (band + 1) * BAND)
            if spread == "band":
                c = rng.choice(hi - lo, n, replace=False)
            elif spread == "window":
                c = 3 * WINDOW + rng.choice(WINDOW, n, replace=False)
            else:       # first and last sub-block of the band
                c = rng.choice(2048, n, replace=False)
                c = np.where(c < 1024, c, BAND - 2048 + c)
            cols.append(lo + c)
        cols = np.sort(np.concatenate(cols))
        row = []
        for i in range(parts):
            keep = cols if i == 0 else cols[rng.random(cols.size) < 0.5]
            row.append(len(brows))
            brows.append(keep)
        arows.append(row)
    def csr(lists):
        ptr = np.zeros(len(lists) + 1, dtype=np.int32)
        np.cumsum([len(x) for x in lists], out=ptr[1:])
        idx = np.concatenate(lists).astype(np.int32)
        return ptr, idx, rng.uniform(-1, 1, idx.size)
    A, B = csr(arows), csr(brows)
    m, n = len(arows), len(brows)
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    h.set_tuning({"row_bins": (0, 0, 0)})        # every row a big row
    h.set_item_order(0)                          # in column order
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for budget in (-1, 0):                       # with a block-pointer table, without
        h.set_block_pointer_budget(budget)
        assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()
