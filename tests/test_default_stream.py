"""Handles made on torch's default stream share one stream per device: the
results of one are the operands of another, and torch hands the memory of a
dropped result to the next, so their kernels have to run in turn."""
from __future__ import annotations

import contextlib
import types

import numpy as np
import pytest

import tilespgemm_amd as tsg


class _Lib:
    """The calls that set a handle's stream, without a GPU."""

    def __init__(self):
        self.handles, self.streams, self.stream_of = 0, 0, {}

    def tsg_create(self, h, device):
        self.handles += 1
        h._obj.value = 0x1000 + self.handles
        return 0

    def hipStreamCreate(self, s):
        self.streams += 1
        s._obj.value = 0x2000 + self.streams
        return 0

    def tsg_set_stream(self, h, s):
        self.stream_of[h.value] = s.value
        return 0

    def __getattr__(self, name):
        if name.startswith("tsg_"):
            return lambda *a: 0
        raise AttributeError(name)


class _Handle(tsg.Handle):
    def __del__(self):                           # may outlive the fake library
        pass


@pytest.fixture
def fake(monkeypatch):
    import torch
    lib = _Lib()
    now = types.SimpleNamespace(cuda_stream=0)
    monkeypatch.setattr(tsg, "load", lambda: lib)
    monkeypatch.setattr(tsg, "_default_streams", {}, raising=False)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: now)
    return lib, now


def _stream(lib, h):
    return lib.stream_of.get(h._h.value)


def test_handles_on_the_default_stream_share_one(fake):
    lib, now = fake
    a, b, other = _Handle(0), _Handle(0), _Handle(1)
    assert _stream(lib, a) and _stream(lib, a) == _stream(lib, b)
    assert _stream(lib, other) not in (None, _stream(lib, a))
    assert lib.streams == 2                      # one a device, however many handles
    a.close()
    assert _stream(lib, _Handle(0)) == _stream(lib, b)


def test_a_stream_of_the_callers_is_used_as_it_is(fake):
    lib, now = fake
    h = _Handle(0)
    shared = _stream(lib, h)
    now.cuda_stream = 0x77
    assert _stream(lib, _Handle(0)) == 0x77
    h.set_stream(now)
    assert _stream(lib, h) == 0x77
    h.set_stream(None)
    assert _stream(lib, h) == shared
    h.set_stream(types.SimpleNamespace(cuda_stream=0))
    assert _stream(lib, h) == shared


@pytest.mark.gpu
def test_two_handles_in_turn_on_the_default_stream():
    """Results dropped at once, and one handle's result as the other's operand."""
    from oracle import py_oracle as O
    from tilespgemm_amd import gen
    n = 3000
    A = gen.erdos_renyi(n, 9.0, seed=4)
    T = gen.transpose(n, n, *A)
    AT = O.csr_spgemm(n, n, A, T)
    want = O.csr_spgemm(n, n, tuple(np.asarray(x, t) for x, t in
                                    zip(AT, (np.int32, np.int32, np.float64))), A)
    one, two = tsg.Handle(0), tsg.Handle(0)
    dA = tsg.DeviceCsr.from_host(n, n, *A)
    for _ in range(10):
        one.spgemm(dA, dA)
        dT = two.transpose(dA)
        ic, jc, c = one.spgemm(dA, dT)
        P = tsg.DeviceCsr(n, n, ic.int(), jc, c)
        got = [x.cpu().numpy() for x in two.spgemm(P, dA)]
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, w)
    one.close()
    two.close()
