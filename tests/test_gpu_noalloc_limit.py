"""tsg_spgemm_noalloc's limit on sizes, from both sides: what it says is what
it applies, and a product at the limit is served."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg

pytestmark = pytest.mark.gpu

SCRATCH = 64 << 20


def _call(h, m, entries):
    """A: m rows, the last entries of them with one; B: 8 columns, one row."""
    import torch
    ptr = np.zeros(m + 1, np.int32)
    ptr[m - entries:] = np.arange(entries + 1)
    A = tsg.DeviceCsr.from_host(m, 1, ptr, np.zeros(entries), np.full(entries, 2.0))
    B = tsg.DeviceCsr.from_host(1, 8, [0, 1], [5], [3.0])
    ic = torch.empty(m + 1, dtype=torch.int64, device="cuda:0")
    jc = torch.empty(entries, dtype=torch.int32, device="cuda:0")
    c = torch.empty(entries, dtype=torch.float64, device="cuda:0")
    assert h.spgemm_noalloc(A, B, ic, jc, c) == entries
    return ptr, ic.cpu().numpy(), jc.cpu().numpy(), c.cpu().numpy()


@pytest.mark.parametrize("method", [tsg.METHOD_AUTO, tsg.METHOD_ROW])
@pytest.mark.parametrize("entries", [1, 1_000_000])
def test_the_limit(entries, method):
    h = tsg.Handle(0, method=method)
    m = (SCRATCH - 8 * (entries + 1)) // 28 - 1           # the most rows served
    ptr, ic, jc, c = _call(h, m, entries)
    np.testing.assert_array_equal(ic, ptr)
    assert (jc == 5).all() and (c == 6.0).all()
    with pytest.raises(tsg.TsgError) as e:
        _call(h, m + 1, entries)
    assert e.value.code == -1 and f"28 (m + 1) + 8 (nnz(A) + 1) <= {SCRATCH}" in str(e.value)
    h.close()
