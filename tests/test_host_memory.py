"""Pinned arrays (lbmpy_amd/host_memory.py) over a stand-in for the GPU's allocation: memory that a forked process does not
inherit, as the driver's mappings are."""
import ctypes
import gc
import os

import numpy as np
import pytest

from lbmpy_amd import _native as nat, host_memory

MADV_DONTFORK = 10


class _Library:
    """lbm355_host_alloc and lbm355_host_free on anonymous memory that is not copied on fork."""

    def __init__(self):
        self.allocated, self.freed, self.refuse = {}, [], False

    def lbm355_host_alloc(self, nbytes):
        if self.refuse or nbytes <= 0:
            return None
        p = host_memory._libc.mmap(None, host_memory._pages(nbytes), 3, 0x22, -1, 0)
        assert host_memory._libc.madvise(ctypes.c_void_p(p), ctypes.c_size_t(host_memory._pages(nbytes)), MADV_DONTFORK) == 0
        self.allocated[p] = nbytes
        return p

    def lbm355_host_free(self, p):
        self.freed.append(p)
        return host_memory._libc.munmap(p, host_memory._pages(self.allocated[p]))


@pytest.fixture
def lib(monkeypatch):
    library = _Library()
    monkeypatch.setattr(nat, "load", lambda *a: library)
    return library


def _in_child(f):
    """What f returns in a forked process."""
    r, w = os.pipe()
    child = os.fork()
    if child == 0:
        status = 1
        try:
            os.write(w, repr(f()).encode())
            status = 0
        finally:
            os._exit(status)
    os.close(w)
    got = os.read(r, 1000).decode()
    os.close(r)
    assert os.waitpid(child, 0)[1] == 0
    return got


def test_exact_size_and_given_back(lib):
    a = host_memory.pinned_array((20, 9, 7))
    assert a.shape == (20, 9, 7) and a.dtype == np.float64 and a.flags.writeable and a.flags.c_contiguous
    assert list(lib.allocated.values()) == [8 * 20 * 9 * 7]
    view = a[3:, 2]
    view[...] = 4.0
    del a
    gc.collect()
    assert not lib.freed and float(view.sum()) == 4.0 * view.size
    del view
    gc.collect()
    assert lib.freed == list(lib.allocated)
    lib.refuse = True
    assert host_memory.pinned_array((3,)) is None


def test_a_forked_process_has_its_own_copy(lib):
    a, b = host_memory.pinned_array((700, 3)), host_memory.pinned_array((5,))
    a[...] = np.arange(2100.0).reshape(700, 3)
    b[...] = 7.0

    def child():
        seen = (float(a.sum()), b.tolist())
        a[...] = 1.0                       # its own
        nested = float(_in_child(lambda: float(a.sum())))
        return seen, nested

    assert eval(_in_child(child)) == ((2100 * 2099 / 2, [7.0] * 5), 2100.0)
    assert float(a.sum()) == 2100 * 2099 / 2
    for _ in range(3):                     # a fork after the other, of changed values
        a += 1
        assert float(_in_child(lambda: float(a.sum()))) == float(a.sum())
    assert not lib.freed


def test_a_forked_process_frees_no_pinned_memory(lib):
    arrays = [host_memory.pinned_array((1000,))]

    def child():
        arrays.clear()
        gc.collect()
        return lib.freed, len(host_memory._inherited)
    assert eval(_in_child(child)) == ([], 0)
    assert not lib.freed and float(arrays[0].sum()) == 0.0
    arrays.clear()
    gc.collect()
    assert lib.freed == list(lib.allocated)


def test_nothing_is_freed_during_a_capture_or_a_fork(lib, monkeypatch):
    a, b, c = (host_memory.pinned_array((n,)) for n in (3, 4, 5))
    with monkeypatch.context() as m:
        m.setattr(host_memory.torch.cuda, "is_initialized", lambda: True)
        m.setattr(host_memory.torch.cuda, "is_current_stream_capturing", lambda: True)
        del a
        gc.collect()
        assert not lib.freed
    with host_memory._forking:
        del b
        gc.collect()
        assert not lib.freed
    del c
    gc.collect()
    assert [lib.allocated[p] for p in lib.freed] == [24, 32, 40]
