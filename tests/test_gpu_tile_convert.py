"""Tile path conversion around its staging limit: a block stages 4 tile rows
(64 rows) of at most 4096 entries in LDS and walks longer ones in memory."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 257])
@pytest.mark.parametrize("width", [1, 63, 64, 65, 96])
def test_blocks_around_the_stage(rows, width):
    """Every row holds width consecutive columns from a random start, so 64
    rows hold 64 * width entries: below, at and above the stage."""
    rng = np.random.default_rng(1000 * rows + width)
    n = rows + width + 16
    start = np.sort(rng.integers(0, n - width + 1, rows))
    ptr = np.concatenate([width * np.arange(rows + 1), np.full(n - rows, width * rows)])
    idx = (start[:, None] + np.arange(width)).ravel().astype(np.int32)
    A = (ptr.astype(np.int32), idx, rng.uniform(-1, 1, idx.size))
    want = O.csr_spgemm(n, n, A, A, fused=True)
    h = tsg.Handle(0, method=tsg.METHOD_TILE, fp_mode=tsg.FP_FUSED)
    dA = tsg.DeviceCsr.from_host(n, n, *A)
    assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dA)], want)
    h.close()
