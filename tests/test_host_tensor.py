"""Who owns a device allocation: copies of tensors on a heap that stands in for the device, without a GPU."""

import copy
import ctypes as C
import gc
import pickle

import numpy as np
import pytest

import lucid_amd as L
from lucid_amd import _C, _tensor as T


class Heap:
    """``lq_alloc`` / ``lq_free`` and the copies, on host memory; a freed block goes to the next request of its size."""

    def __init__(self):
        self.live, self.idle, self.freed_twice = {}, [], []

    def call(self, name, *args):
        if name == "lq_alloc":
            out, n = args
            block = next((b for b in self.idle if len(b) == max(n, 1)), None)
            if block is None:
                block = C.create_string_buffer(max(n, 1))
            else:
                self.idle.remove(block)
            self.live[C.addressof(block)] = block
            out._obj.value = C.addressof(block)
        elif name in ("lq_h2d", "lq_d2h", "lq_d2d"):
            C.memmove(*args[:3])
        else:
            raise AssertionError(name)

    def lq_free(self, ptr):
        block = self.live.pop(ptr, None)
        if block is None:
            self.freed_twice.append(ptr)
        else:
            self.idle.append(block)


@pytest.fixture
def heap(monkeypatch):
    h = Heap()
    gc.collect()
    monkeypatch.setattr(_C, "call", h.call)
    monkeypatch.setattr(_C, "load", lambda: h)
    monkeypatch.setattr(_C, "_initialised_device", 0)
    yield h
    gc.collect()  # (what the test made is freed here)


@pytest.mark.parametrize("copied", [lambda t: pickle.loads(pickle.dumps(t)), copy.copy, copy.deepcopy])
@pytest.mark.parametrize("view", [False, True])
@pytest.mark.parametrize("n", [0, 24])
def test_a_dropped_copy_leaves_the_tensor_alone(heap, copied, view, n):
    a = np.arange(n, dtype=np.float32).reshape(n // 3, 3)
    t = L.tensor(a, device="hip")
    if view:
        t, a = t.narrow_rows(n // 6), a[:n // 6]
    c = copied(t)
    assert np.array_equal(c.numpy(), a) and c.dtype == t.dtype and c.shape == t.shape
    del c
    gc.collect()
    other = T.Tensor.from_numpy(np.full((n // 3, 3), 7, np.float32))  # takes whatever was given back
    assert np.array_equal(t.numpy(), a)
    del t, other
    gc.collect()
    assert heap.freed_twice == [] and heap.live == {}


def test_a_copied_buffer_is_another_allocation(heap):
    b = T.DeviceBuffer(8)
    C.memmove(b.ptr, b"lucidamd", 8)
    for c in (copy.copy(b), copy.deepcopy(b), pickle.loads(pickle.dumps(b))):
        assert c.ptr != b.ptr and c.nbytes == 8 and C.string_at(c.ptr, 8) == b"lucidamd"
