"""Row path, rows of at most 1024 products (tsg_flat.h): products at the edges
of the kernels' register counts, more than 64 A entries in a row, spans past
one column window, B rows of one entry (many B rows per batch), repeated B
columns, and outputs past one accumulation pass -- bitwise against the oracle
in both FP modes."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 48, 49, 63, 64, 65, 191, 192, 193, 255, 256, 257, 384, 385, 511, 512, 513,
         767, 768, 769, 1023, 1024, 1025]
LENGTHS = [0, 1, 2, 3, 5, 17, 27, 64, 65, 130, 256]


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate([np.asarray(x, dtype=np.int32) for x in lists])
    return ptr, idx, rng.uniform(-1, 1, idx.size)


def _operands(shape, span, repeat, seed):
    """B: 40 rows of every length in LENGTHS with columns over span columns
    that start off a word boundary (repeat: one column twice in every longer
    row); A: for every edge, rows whose B rows' lengths add up to it."""
    rng = np.random.default_rng(seed)
    k = 3_000_000
    brows = []
    for n in LENGTHS:
        for _ in range(40):
            cols = np.sort(rng.choice(max(span, n), n, replace=False)) + 1237
            if repeat and n > 2:
                cols[1] = cols[0]
            brows.append(cols)
    arows = []
    sizes = {"long": LENGTHS, "short": [0, 1, 2, 3]}[shape]
    for total in EDGES:
        for _ in range(3):
            row, left = [], total
            while left > 0:
                n = int(rng.choice([x for x in sizes if x <= left]))
                row.append(LENGTHS.index(n) * 40 + int(rng.integers(40)))
                left -= n
            arows.append(row)
    A, B = _csr(arows, rng), _csr(brows, rng)
    return len(arows), len(brows), k, A, B


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("span", [300, 30_000, 2_900_000])
@pytest.mark.parametrize("shape", ["long", "short"])
def test_flat_rows_at_their_edges(shape, span, repeat, fp):
    m, n, k, A, B = _operands(shape, span, repeat, seed=span + repeat)
    fused = fp == tsg.FP_FUSED
    want = O.csr_spgemm(m, k, A, B, fused=fused)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for bins in ((64, 256, 1024), (0, 0, 1024), (16, 256, 700)):
        h.set_tuning({"row_bins": bins})
        got = [x.cpu().numpy() for x in h.spgemm(dA, dB)]
        assert_csr_equal(got, want)
    h.close()
