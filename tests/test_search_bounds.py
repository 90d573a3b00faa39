"""The kernels' binary search at positions near the largest that an int32
CSR can have: built for the host from the header the kernels include and run
over 2^31 - 1 entries, all zero pages that are never touched but for the
probes."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from tilespgemm_amd import build

SOURCE = r"""
#include "tsg_device.h"
extern "C" int search(const int *a, int lo, int hi, int key) {
    return lower_bound_i32(a, lo, hi, key);
}
"""
LAST = 2**31 - 1


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    d = tmp_path_factory.mktemp("search")
    src, lib = os.path.join(d, "search.hip"), os.path.join(d, "libsearch.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([build.hipcc(), *build.flags(), "--offload-host-only", "-I", build.CSRC,
                    "-shared", src, "-o", lib], check=True, capture_output=True)
    f = C.CDLL(lib).search
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int]
    return f


@pytest.fixture(scope="module")
def zeros():
    return np.zeros(LAST, dtype=np.int32)


@pytest.mark.parametrize("lo,hi", [(0, LAST), (0, 2**30 + 1), (2**30, 2**30 + 1),
                                   (2**30 - 1, LAST), (LAST - 1, LAST), (LAST, LAST), (5, 5)])
def test_every_probe_is_in_range(search, zeros, lo, hi):
    at = zeros.ctypes.data
    assert search(at, lo, hi, 1) == hi           # past all of them
    assert search(at, lo, hi, 0) == lo           # before all of them


def test_a_step_near_the_end(search, zeros):
    zeros[LAST - 3:] = 7
    assert search(zeros.ctypes.data, 0, LAST, 7) == LAST - 3
    zeros[LAST - 3:] = 0
