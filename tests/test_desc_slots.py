"""The descriptors that a thread's flash-attention calls reuse: what a slot
holds always matches the tensor last given, whatever it held before (no GPU)."""
import ctypes
import threading

import pytest
import torch

import tecoops
from tecoops import _lib


def held(d):
    dt, n = ctypes.c_int(), ctypes.c_int()
    dims, strides = (ctypes.c_int * 16)(), (ctypes.c_int * 16)()
    _lib.call("tecoopsGetTensorNdDescriptor", d, 16, ctypes.byref(dt), ctypes.byref(n), dims, strides)
    return dt.value, tuple(dims[:n.value]), tuple(strides[:n.value])


BASE = torch.empty(6, 4, 8, 16)


@pytest.mark.parametrize("order", [(0, 1, 2, 3, 4, 5), (3, 0, 3, 1, 5, 5, 2, 4, 0)])
def test_slot_follows_the_tensor(order):
    forms = [(BASE, _lib.DATA_HALF), (BASE, _lib.DATA_BFLOAT16), (BASE[:3], _lib.DATA_HALF),
             (BASE.transpose(0, 1), _lib.DATA_HALF), (BASE[:, :, 0], _lib.DATA_HALF),
             (torch.empty([1] * 11 + [3]), _lib.DATA_INT32)]  # past the fixed-size arrays
    slots = tecoops._DescSlots(2)
    for i in order:
        t, code = forms[i]
        for _ in range(2):
            assert held(slots.fill(1, t, code)) == (code, tuple(t.shape), t.stride())
        assert held(slots.fill(0, BASE, _lib.DATA_HALF))[1] == tuple(BASE.shape)


def test_refused_tensor_leaves_nothing_held():
    slots = tecoops._DescSlots(1)
    slots.fill(0, BASE, _lib.DATA_HALF)
    for _ in range(2):
        with pytest.raises(_lib.TecoopsError) as e:
            slots.fill(0, torch.empty(()), _lib.DATA_HALF)
        assert e.value.status == _lib.BAD_PARAM
    assert held(slots.fill(0, BASE, _lib.DATA_HALF))[1] == tuple(BASE.shape)


def test_threads_have_slots_of_their_own():
    mine, other = tecoops._desc_slots(), []
    th = threading.Thread(target=lambda: other.append(tecoops._desc_slots()))
    th.start()
    th.join()
    assert tecoops._desc_slots() is mine and other[0] is not mine
