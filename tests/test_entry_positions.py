"""The positions of a row's entries that the row path's pipeline loads, for
rows at the end of the largest array an int32 CSR can have: every entry once,
in order, and nothing outside the row however far ahead is looked.  Built for
the host from the header the kernels include."""
from __future__ import annotations

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from tilespgemm_amd import build

SOURCE = r"""
#include "tsg_internal.h"
#include "tsg_expand.h"
extern "C" int at(unsigned g, unsigned pe, int parts, int part, int lane) {
    int p;
    const bool in = parts == 1 ? entry_at<1>(g, pe, part, lane, p)
                               : entry_at<2>(g, pe, part, lane, p);
    return in ? p : -1;
}
"""
LAST = 2**31 - 1


@pytest.fixture(scope="module")
def at(tmp_path_factory):
    d = tmp_path_factory.mktemp("entries")
    src, lib = os.path.join(d, "entries.hip"), os.path.join(d, "libentries.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([build.hipcc(), *build.flags(), "--offload-host-only", "-I", build.CSRC,
                    "-shared", src, "-o", lib], check=True, capture_output=True)
    f = C.CDLL(lib).at
    f.argtypes = [C.c_uint, C.c_uint, C.c_int, C.c_int, C.c_int]
    return f


@pytest.mark.parametrize("parts", [1, 2])
@pytest.mark.parametrize("pe", [LAST, LAST - 1, LAST - 63, 2**30 + 5, 200])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 200])
def test_a_row_and_what_is_looked_at_ahead(at, parts, pe, n):
    pa, seen = pe - n, []
    g = pa
    while g < pe:                                 # as the kernels' loops, in 32 bits
        for lane in range(64):
            for part in range(parts):
                for ahead in range(4):
                    p = at((g + ahead * 64 * parts) % 2**32, pe, parts, part, lane)
                    assert p == -1 or pa <= p < pe
                    if ahead == 0 and p >= 0:
                        seen.append(p)
        g = (g + 64 * parts) % 2**32
    assert seen == list(range(pa, pe))
