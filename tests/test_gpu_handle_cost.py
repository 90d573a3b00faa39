"""Making and closing a handle costs the same whether or not another one is
open: what a device's handles share is kept."""
from __future__ import annotations

import gc
import time

import pytest

import tilespgemm_amd as tsg

pytestmark = pytest.mark.gpu


def _cost(rounds=60):
    took = []
    for _ in range(rounds):
        t0 = time.perf_counter()
        tsg.Handle(0).close()
        took.append(time.perf_counter() - t0)
    return sorted(took)[rounds // 2]


def test_the_only_handle_costs_no_more():
    gc.collect()
    tsg.Handle(0).close()
    alone = _cost()
    other = tsg.Handle(0)
    beside = _cost()
    other.close()
    assert alone < 1.5 * beside, (alone, beside)


def test_more_handles_than_the_slab_holds():
    """Boxes past the slab's 64, closed in another order than made."""
    import numpy as np
    from oracle import py_oracle as O
    from tilespgemm_amd import gen
    A = gen.erdos_renyi(300, 5.0, seed=3)
    want = O.csr_spgemm(300, 300, A, A)
    dA = tsg.DeviceCsr.from_host(300, 300, *A)
    for _ in range(2):
        handles = [tsg.Handle(0) for _ in range(70)]
        for h in handles[::3] + handles[1::3] + handles[2::3]:
            ic, jc, c = h.spgemm(dA, dA)
            np.testing.assert_array_equal(ic.cpu().numpy(), want[0])
            np.testing.assert_array_equal(c.cpu().numpy(), want[2])
            h.close()
