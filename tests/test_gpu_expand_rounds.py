"""The big rows' product expansion (expand_group): a group of 64 A entries goes
through its products in rounds of up to 8 batches of 64, a short rest in rounds
of half or a quarter.  Rows whose group totals lie around every round's end,
with entries that start on it, go over it, span whole rounds or are empty, in
every kernel that expands -- bands, dense, sparse and hash items -- against the
oracle in both FP modes."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 31, 32, 63, 64, 65, 127, 128, 129, 256, 384, 511, 512, 513, 1100]
TOTALS = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 383, 384, 385, 511, 512, 513,
          576, 639, 640, 641, 767, 768, 769, 1023, 1024, 1025, 1536, 3000]


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate(lists).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("span", [1200, 9000, 60_000])   # dense, mixed and sparse items
@pytest.mark.parametrize("order", [0, 1 << 60])
def test_totals_around_the_rounds(span, order, fp):
    rng = np.random.default_rng(span)
    k, copies = 131_072, 30
    brows = [np.sort(rng.choice(span, min(n, span), replace=False)) + 517
             for n in LENGTHS for _ in range(copies)]
    at = {n: i * copies for i, n in enumerate(LENGTHS)}
    arows = []
    for total in TOTALS:
        for most in (1, 64, 513, 1100):              # the longest entry that is taken
            row, left = [], total
            while left > 0 and len(row) < 200:
                n = int(rng.choice([x for x in LENGTHS if x <= min(left, most)]))
                row.append(at[n] + int(rng.integers(copies)))
                left -= n
            arows.append(np.array(row))               # in no order: so are its products
    # the second of two groups starts where the first one's rounds end
    arows.append(np.concatenate([np.full(64, at[64]) + np.arange(64) % copies,
                                 np.full(64, at[65]) + np.arange(64) % copies]))
    A, B = _csr(arows, rng), _csr(brows, rng)
    m, n = len(arows), len(brows)
    want = O.csr_spgemm(m, k, A, B, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    h.set_tuning({"row_bins": (0, 0, 0)})            # every row a big row
    h.set_item_order(order)
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for pointers in (6 << 30, 0):
        for bitmap in (-1, 0):
            h.set_block_pointer_budget(pointers)
            h.set_bitmap_budget(bitmap)
            assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()
