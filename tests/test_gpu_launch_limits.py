"""Work for more threads than one launch holds (2^32) away from the short rows:
2^26 big rows with their bands and items, block pointers of a B of 2^26 rows,
2^26 work units of the tile path."""
from __future__ import annotations

import numpy as np
import pytest

import tilespgemm_amd as tsg

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
OVER = (1 << 26) + 70


def _range(n):
    import torch
    return torch.arange(n, dtype=torch.int32, device=DEV)


def _values(n, seed=1):
    import torch
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand(n, dtype=torch.float64, device=DEV, generator=g)


@pytest.mark.parametrize("order", [0, 1 << 60])
def test_big_rows(order):
    """One entry a row, every row a big row, of B's 5 rows of one entry."""
    import torch
    m = OVER
    a = _values(m)
    A = tsg.DeviceCsr(m, 5, _range(m + 1), _range(m) % 5, a)
    cols, b = np.array([3, 0, 1, 4, 4], np.int32), np.array([2.0, -1.0, 0.5, 4.0, -8.0])
    B = tsg.DeviceCsr.from_host(5, 6, np.arange(6), cols, b)
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    h.set_tuning({"row_bins": (0, 0, 0)})
    h.set_item_order(order)
    ic, jc, c = h.spgemm(A, B)
    at = (_range(m) % 5).long()
    assert torch.equal(ic, torch.arange(m + 1, dtype=torch.int64, device=DEV))
    assert torch.equal(jc, torch.from_numpy(cols).to(DEV)[at])
    assert torch.equal(c, a * torch.from_numpy(b).to(DEV)[at])
    h.close()


def test_block_pointers_of_many_rows():
    """Two big rows that name the first and last rows of B."""
    import torch
    n = OVER
    named = torch.cat([_range(1500), n - 1500 + _range(1500)])
    a, b = _values(6000, 2), _values(n, 3)
    A = tsg.DeviceCsr(2, n, torch.tensor([0, 3000, 6000], dtype=torch.int32, device=DEV),
                      torch.cat([named, named]), a)
    B = tsg.DeviceCsr(n, 5000, _range(n + 1), _range(n) % 5000, b)
    h = tsg.Handle(0, method=tsg.METHOD_ROW)
    h.set_block_pointer_budget(6 << 30)
    ic, jc, c = h.spgemm(A, B)
    want = torch.zeros(2, 5000, dtype=torch.float64, device=DEV)
    hit = torch.zeros(2, 5000, dtype=torch.bool, device=DEV)
    for r in range(2):                           # in order; no column more than twice
        for half in (slice(0, 1500), slice(1500, 3000)):
            col = (named[half] % 5000).long()
            v = a[3000 * r:3000 * (r + 1)][half]
            want[r, col] = torch.addcmul(want[r, col], v, b[named[half].long()])
            hit[r, col] = True
    assert ic.tolist() == [0, int(hit[0].sum()), int(hit.sum())]
    assert torch.equal(jc.long(), hit.nonzero()[:, 1])
    torch.testing.assert_close(c, want[hit], rtol=1e-15, atol=0)
    h.close()


def test_units_of_the_tile_path():
    """2^28 rows of one entry times a dense 16 x 16 B: every 16 x 16 tile of C is
    full, four units of 64 outputs each."""
    import torch
    m = (1 << 28) + 48
    a = _values(m, 4)
    A = tsg.DeviceCsr(m, 16, _range(m + 1), _range(m) % 16, a)
    b = _values(256, 5)
    B = tsg.DeviceCsr(16, 16, 16 * _range(17), _range(256) % 16, b)
    h = tsg.Handle(0, method=tsg.METHOD_TILE)
    ic, jc, c = h.spgemm(A, B)
    h.close()
    assert int(ic[-1]) == 16 * m == c.numel()
    step = 1 << 22
    for r in range(0, m, step):
        e = min(m, r + step)
        row = torch.arange(r, e, device=DEV)
        assert torch.equal(ic[r:e], 16 * row)
        assert bool((jc[16 * r:16 * e].view(-1, 16) == _range(16)).all())
        assert torch.equal(c[16 * r:16 * e].view(-1, 16),
                           a[r:e, None] * b.view(16, 16)[row % 16])
