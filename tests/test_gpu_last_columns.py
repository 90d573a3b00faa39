"""Big rows of matrices with as many columns as an int32 allows: outputs in the
last sub-block, whose end does not fit an int, in rows' and column order, with
and without the bitmaps and block pointers, against the oracle on columns
relabelled in order."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import tilespgemm_amd as tsg
from oracle import py_oracle as O
from tests.util import assert_csr_equal
from tilespgemm_amd import build

SOURCE = r"""
#include "tsg_internal.h"
extern "C" int start(int sb, int k) { return sub_block_start(sb, k); }
"""


def test_ends_of_sub_blocks(tmp_path):
    src, lib = os.path.join(tmp_path, "sub.hip"), os.path.join(tmp_path, "libsub.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([build.hipcc(), *build.flags(), "--offload-host-only", "-I", build.CSRC,
                    "-shared", src, "-o", lib], check=True, capture_output=True)
    start = C.CDLL(lib).start
    for k in (1, 1024, 1025, 2**30, 2**31 - 1024, 2**31 - 1023, 2**31 - 1):
        for sb in {0, 1, k >> 10, (k + 1023) >> 10}:
            assert start(sb, k) == min(k, sb * 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [2**31 - 1, 2**31 - 1023, 2**31 - 1024, 2**30 + 1])
@pytest.mark.parametrize("order", [0, 1 << 60])
def test_big_rows_with_outputs_in_the_last_columns(k, order):
    rng = np.random.default_rng(k % 97)
    near = np.unique(k - 1 - rng.integers(0, 3000, 900))
    far = np.unique(rng.integers(0, k, 900))
    brows = [np.array([k - 1]), near, far, np.unique(np.concatenate([near[-200:], far[:50]])),
             np.arange(k - 70, k), np.array([0, k - 1])]
    arows = [np.arange(6), np.array([0]), np.array([1, 2]), np.array([4, 5]), np.array([3])]

    def csr(lists):
        ptr = np.zeros(len(lists) + 1, dtype=np.int32)
        np.cumsum([len(x) for x in lists], out=ptr[1:])
        idx = np.concatenate(lists).astype(np.int32)
        return ptr, idx, rng.uniform(-1, 1, idx.size)

    A, B = csr(arows), csr(brows)
    used, at = np.unique(B[1], return_inverse=True)
    ic, jc, c = O.csr_spgemm(5, used.size, A, (B[0], at.astype(np.int32), B[2]))
    want = (ic, used[jc].astype(np.int32), c)
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    h.set_tuning({"row_bins": (0, 0, 0)})
    h.set_item_order(order)
    dA, dB = tsg.DeviceCsr.from_host(5, 6, *A), tsg.DeviceCsr.from_host(6, k, *B)
    for pointers in (-1, 0, 1 << 20):
        for bitmap in (-1, 0):
            h.set_block_pointer_budget(pointers)
            h.set_bitmap_budget(bitmap)
            assert_csr_equal([x.cpu().numpy() for x in h.spgemm(dA, dB)], want)
    h.close()
