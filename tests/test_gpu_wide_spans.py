"""Row path, short rows whose columns span more than the bitmap's first level
(131,072 columns for rows of up to 64 products, 262,144 for longer ones): the
span's edges, columns at both ends, in clusters over word and block edges, up
to the last column of an int32, against the oracle on columns relabelled in
order -- and the time, which follows the products and not the span."""
from __future__ import annotations

import time

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 63, 64, 65, 200, 256, 257, 511, 513, 1000, 1024, 1025, 1536]
SPANS = [131_056, 131_072, 131_088, 262_128, 262_144, 262_145, 2**20 + 3, 2**24 + 1, 2**30,
         2**31 - 1]


def _columns(kind, k, rng):
    """A pool of columns below k."""
    if kind == "spread":
        c = rng.integers(0, k, 6000)
    elif kind == "ends":
        c = np.concatenate([np.arange(700), k - 1 - np.arange(700)])
    elif kind == "clusters":
        c = (rng.integers(0, k, 150)[:, None] + np.arange(-9, 25)).ravel()
    else:
        edge = np.array([2**s for s in range(4, 32) if 2**s <= k])
        c = (edge[:, None] + edge[None, :] // 2 + np.array([-17, -16, -1, 0, 1, 15])[:, None, None])
        c = np.append(c.ravel(), [0, k - 1])
    c = np.unique(np.append(c, [0, k - 1]))
    return c[(c >= 0) & (c < k)]


def _csr(lists, rng):
    ptr = np.zeros(len(lists) + 1, dtype=np.int32)
    np.cumsum([len(x) for x in lists], out=ptr[1:])
    idx = np.concatenate(lists).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


@pytest.mark.parametrize("fp", [tsg.FP_FUSED, tsg.FP_SEPARATE])
@pytest.mark.parametrize("kind", ["spread", "ends", "clusters", "blocks"])
@pytest.mark.parametrize("k", SPANS)
def test_spans_past_the_first_level(k, kind, fp):
    rng = np.random.default_rng(k % 1000 + len(kind))
    pool = _columns(kind, k, rng)
    arows, brows = [], []
    for total in SIZES:
        for entries in (1, 40, 300):              # 300: more than 64 entries in a row
            cuts = np.sort(rng.integers(0, total + 1, min(entries, total) - 1))
            lens = np.diff(np.concatenate([[0], cuts, [total]]))
            row = []
            for n in lens:
                row.append(len(brows))
                brows.append(np.sort(rng.choice(pool, min(int(n), pool.size), replace=False)))
            # both ends of the span in every longer row
            if lens[0] > 1:
                b = brows[row[0]]
                b[0], b[-1] = 0, k - 1
            arows.append(np.array(row))
    m, n = len(arows), len(brows)
    A, B = _csr(arows, rng), _csr(brows, rng)
    used, at = np.unique(B[1], return_inverse=True)
    fused = fp == tsg.FP_FUSED
    ic, jc, c = O.csr_spgemm(m, used.size, A, (B[0], at.astype(np.int32), B[2]), fused=fused)
    want = (ic, used[jc].astype(np.int32), c)
    h = tsg.Handle(0, method=tsg.METHOD_ROW, fp_mode=fp)
    dA, dB = tsg.DeviceCsr.from_host(m, n, *A), tsg.DeviceCsr.from_host(n, k, *B)
    for bins in ((64, 256, 1024), (0, 0, 1024)):
        h.set_tuning({"row_bins": bins})
        assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()


@pytest.mark.parametrize("deg", [8, 14, 30])
def test_time_follows_the_products(deg):
    """Rows of deg * deg products: over 2^28 columns less than 5 times as long
    as over 2^16 (window by window it was 6, 26 and 60 times)."""
    import torch
    rng = np.random.default_rng(deg)
    n = 32768
    ip = np.arange(0, n * deg + 1, deg, dtype=np.int32)

    def matrix(k):
        col = np.sort(rng.integers(0, k, (n, deg)), axis=1)
        return tsg.DeviceCsr.from_host(n, k, ip, col.ravel(), np.ones(n * deg))

    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    A, took = matrix(n), []
    for k in (2**16, 2**28):
        B, best = matrix(k), 1e9
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            h.spgemm(A, B)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        took.append(best)
    h.close()
    assert took[1] < 5 * took[0], took
