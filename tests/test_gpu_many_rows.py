"""More short rows than one launch has threads for: 2^26 rows of 65 products (a
wave each), every product of one column, so that C has one entry a row."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O

pytestmark = pytest.mark.gpu


def test_rows_past_one_launch():
    import torch
    m, each = (1 << 26) + 70, 65
    rng = np.random.default_rng(3)
    B = (np.array([0, each], np.int32), np.full(each, 2, np.int32), rng.uniform(-1, 1, each))
    one = (np.array([0, 1], np.int32), np.zeros(1, np.int32), np.array([0.75]))
    want = O.csr_spgemm(1, 4, one, B)
    dev = "cuda:0"
    A = tsg.DeviceCsr(m, 1, torch.arange(m + 1, dtype=torch.int32, device=dev),
                      torch.zeros(m, dtype=torch.int32, device=dev),
                      torch.full((m,), 0.75, dtype=torch.float64, device=dev))
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    ic, jc, c = h.spgemm(A, tsg.DeviceCsr.from_host(1, 4, *B))
    assert torch.equal(ic, torch.arange(m + 1, dtype=torch.int64, device=dev))
    assert bool((jc == 2).all())
    assert bool((c == want[2][0]).all())
    h.close()
