"""The first pass over a product's operands (tsg_front.hip): input checks,
products per row and row bins over blocks of 1024 and 4096 items (a row's
entries, then its end).  Rows that end or start on a block's edge, rows over
many blocks, long runs of empty rows, and faults placed on the edges."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal

pytestmark = pytest.mark.gpu


def _matrix(lens, ncols, seed):
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens)
    ptr = np.zeros(lens.size + 1, dtype=np.int32)
    np.cumsum(lens, out=ptr[1:])
    idx = np.concatenate([np.sort(rng.choice(ncols, n, replace=False)) for n in lens if n] or
                         [np.zeros(0)]).astype(np.int32)
    return ptr, idx, rng.uniform(-1, 1, idx.size)


SHAPES = {
    # a row and its end fill a block exactly, one entry less, one more
    "edges": [1023, 1022, 1, 1024, 1023, 0, 4, 1018, 2047],
    # one row over several blocks between short ones
    "long": [3] * 40 + [9000] + [2] * 40 + [0, 0, 5000],
    # runs of empty rows over whole blocks, entries at both ends
    "empty": [5] + [0] * 5000 + [7, 1] + [0] * 2500,
    "none": [0] * 1500,
    "one": [1],
}


@pytest.mark.parametrize("blocks", ["small", "large"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_rows_over_block_edges(shape, blocks):
    n = 9500
    lens = list(SHAPES[shape])
    if blocks == "large":
        # more than 2^20 items: blocks of 4096 items
        lens = lens * 3 + [0] * (1 << 20) + lens
    A = _matrix(lens, n, seed=len(lens))
    B = _matrix([(i * 7) % 5 for i in range(n)], 4000, seed=2)
    m = len(lens)
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    got = [x.cpu().numpy() for x in h.spgemm(tsg.DeviceCsr.from_host(m, n, *A),
                                             tsg.DeviceCsr.from_host(n, 4000, *B))]
    h.close()
    assert_csr_equal(got, O.csr_spgemm(m, 4000, A, B))


@pytest.mark.parametrize("at", [0, 1022, 1023, 1024, 2046, 4999])
def test_faults_on_block_edges_are_seen(at):
    """One bad column, one entry out of order inside a row, and one row
    pointer out of order, at entries around the blocks' edges."""
    n = 6000
    A = _matrix([5000, 400, 0, 300], n, seed=1)
    B = _matrix([1] * n, 50, seed=2)
    dB = tsg.DeviceCsr.from_host(n, 50, *B)
    h = tsg.Handle(0)
    for bad in (-1, n):
        X = (A[0], A[1].copy(), A[2])
        X[1][at] = bad
        with pytest.raises(tsg.TsgError) as e:
            h.spgemm(tsg.DeviceCsr.from_host(4, n, *X), dB)
        assert e.value.code == -1 and "column out of range" in str(e.value)
    X = (np.array([0, at + 1, at, 5400, 5700], np.int32), A[1], A[2])
    with pytest.raises(tsg.TsgError) as e:
        h.spgemm(tsg.DeviceCsr.from_host(4, n, *X), dB)
    assert e.value.code == -1 and "row pointers" in str(e.value)
    # out of order: refused where sorted rows are needed, served by the row path
    X = (A[0], A[1].copy(), A[2])
    i = max(at, 1)
    X[1][[i - 1, i]] = X[1][[i, i - 1]]
    dX = tsg.DeviceCsr.from_host(4, n, *X)
    h.set_method(tsg.METHOD_TILE)
    with pytest.raises(tsg.TsgError) as e:
        h.spgemm(dX, dB)
    assert e.value.code == -1 and "sorted" in str(e.value)
    h.set_method(tsg.METHOD_AUTO)
    got = [x.cpu().numpy() for x in h.spgemm(dX, dB)]
    assert h.method_used == tsg.METHOD_ROW
    assert_csr_equal(got, O.csr_spgemm(4, 50, X, B))
    h.close()


def test_more_than_2p32_products_in_a_block():
    """5000 entries of one row on a B row of 2^20 ones: 5.2e9 products from
    two blocks' entries; every output is exactly 5000."""
    k = 1 << 20
    A = (np.array([0, 0, 5000, 5000], np.int32), np.zeros(5000, np.int32), np.ones(5000))
    B = (np.array([0, k], np.int32), np.arange(k, dtype=np.int32), np.ones(k))
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    dA, dB = tsg.DeviceCsr.from_host(3, 1, *A), tsg.DeviceCsr.from_host(1, k, *B)
    ic, jc, c = h.spgemm(dA, dB)
    assert ic.cpu().tolist() == [0, 0, k, k]
    assert np.array_equal(jc.cpu().numpy(), np.arange(k))
    assert np.array_equal(c.cpu().numpy(), np.full(k, 5000.0))
    h.close()
