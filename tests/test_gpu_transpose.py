"""Transpose: column pointers taken from the sorted columns, and the sort's two
kinds of passes (around 204,800 entries), against the host transpose."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from tilespgemm_amd import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [0, 1, 204_799, 204_800, 204_801, 300_000])
@pytest.mark.parametrize("cols", [1, 700, 1_000_003])
def test_transpose_at_the_sorts_edges(nnz, cols):
    rng = np.random.default_rng(nnz + cols)
    m = 5000
    # a third of the entries in one hub column, unsorted rows, empty rows
    idx = rng.integers(0, cols, nnz)
    idx[rng.random(nnz) < 0.33] = cols // 2
    ptr = np.zeros(m + 1, np.int32)
    cuts = np.sort(rng.integers(0, nnz + 1, m - 1))
    ptr[1:m], ptr[m] = cuts, nnz
    val = rng.uniform(-1, 1, nnz)
    h = tsg.Handle(0)
    T = h.transpose(tsg.DeviceCsr.from_host(m, cols, ptr, idx, val))
    want = gen.transpose(m, cols, ptr, idx, val)
    assert np.array_equal(T.indptr.cpu().numpy(), want[0])
    assert np.array_equal(T.indices.cpu().numpy(), want[1])
    assert np.array_equal(T.data.cpu().numpy(), want[2])
    h.close()
