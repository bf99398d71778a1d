"""Tensor arguments of the leaf routines: what the short check accepts is what
the full checks accept, and what it does not accept still raises what they
raise.  With a stand-in for torch, so that no GPU is needed."""
import sys
import types

import numpy as np
import pytest


FLOAT64 = object()


class Tensor:
    def __init__(self, a, cuda=True):
        self.a, self.is_cuda = a, cuda
        self.dtype = FLOAT64 if a.dtype == np.float64 else a.dtype
        self.shape = tuple(a.shape)

    def numel(self):
        return self.a.size

    def dim(self):
        return self.a.ndim

    def stride(self):
        return tuple(s // self.a.itemsize for s in self.a.strides)

    def is_contiguous(self):
        return self.a.flags.c_contiguous

    def data_ptr(self):
        return self.a.ctypes.data


Tensor.__module__ = "torch"
S = (5, 4, 3)  # Fortran shape of the grid


def arrays():
    z = np.zeros
    yield from ((z(60), True), (z(59), True), (z(61), True), (z(120)[::2], True), (z(60), False),
                (z(60, np.float32), True), (z(S[::-1]), True), (z(S), True),
                (z(S, order="F"), True), (z(S[::-1], order="F"), True), (z((3, 5, 4)), True),
                (z((4, 4, 3)), True), (z((6, 10)), True), (z((10, 6), order="F"), True),
                (z((3, 4, 10))[:, :, ::2], True), (z((3, 4, 6)), True), (z((1, 60, 1)), True))


@pytest.mark.parametrize("shape", [None, S])
@pytest.mark.parametrize("k", range(17))
def test_short_check_agrees_with_the_full_one(monkeypatch, k, shape):
    from picsar_amd.picsarpy import _Call
    fake = types.ModuleType("torch")
    fake.Tensor, fake.float64 = Tensor, FLOAT64
    monkeypatch.setitem(sys.modules, "torch", fake)
    a, cuda = list(arrays())[k]
    t = Tensor(a, cuda)

    def outcome(f):
        c = _Call()
        try:
            return f(c), c.torch
        except (TypeError, ValueError) as e:
            return type(e), str(e)

    assert outcome(lambda c: c.arr(t, 60, "x", fortran_shape=shape)) == \
        outcome(lambda c: c._tensor_ptr(t, 60, "x", shape))
