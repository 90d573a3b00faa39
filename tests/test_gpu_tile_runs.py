"""Tile path products taken as runs: bands and blocks whose tiles' products are
consecutive, the same with holes (which are walked), and tiles of both kinds."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu


def _pattern(kind, n, rng):
    i = np.arange(n)
    d = i[None, :] - i[:, None]
    if kind == "band":
        return np.abs(d) <= 16
    if kind == "wide band":
        return np.abs(d) <= 61
    if kind == "one side":
        return (d >= 3) & (d <= 40)
    if kind == "blocks":
        return (i[None, :] // 48) == (i[:, None] // 48)
    if kind == "every other":
        return (np.abs(d) <= 33) & (i[None, :] % 2 == 0)
    if kind == "holes":
        return (np.abs(d) <= 24) & (rng.random((n, n)) < 0.9)
    # runs in one half of the rows, holes in the other
    return (np.abs(d) <= 20) & ((i[:, None] < n // 2) | (rng.random((n, n)) < 0.7))


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("n", [16, 33, 300])
@pytest.mark.parametrize("kind", ["band", "wide band", "one side", "blocks", "every other",
                                  "holes", "mixed"])
def test_runs_and_holes(kind, n, fp):
    rng = np.random.default_rng(n)
    keep = _pattern(kind, n, rng)
    ptr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    idx = np.nonzero(keep)[1].astype(np.int32)
    A = (ptr, idx, rng.uniform(-1, 1, idx.size))
    want = O.csr_spgemm(n, n, A, A, fused=fp == tsg.FP_FUSED)
    h = tsg.Handle(0, method=tsg.METHOD_TILE, fp_mode=fp)
    dA = tsg.DeviceCsr.from_host(n, n, *A)
    assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dA)], want)
    h.close()
