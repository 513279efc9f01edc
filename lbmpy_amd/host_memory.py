"""Pinned host memory for numpy arrays that kernels write directly.

Pinned memory is a mapping of the GPU's driver: it is not inherited by a forked process, and giving it back waits for the
GPU.  So arrays here are freed with their last view, but not on a thread whose stream is being captured, and a process
forked from Python finds its own copy of them at the same addresses.
"""
import collections
import ctypes
import mmap
import os
import threading
import weakref

import numpy as np
import torch

from . import _native as nat

_live = {}                             # address -> bytes of this process's pinned arrays
_inherited = {}                        # the same of the copies that a forked process got
_given_up = collections.deque()        # addresses to free; some wait, after a capture or a fork, for the next array to go
_forking = threading.Lock()            # held during a fork, and while memory is freed
_copies = []

_libc = ctypes.CDLL(None, use_errno=True)
_libc.mmap.restype = _libc.mremap.restype = ctypes.c_void_p
_libc.mmap.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
_libc.mremap.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
_libc.munmap.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
_MAP_FAILED = ctypes.c_void_p(-1).value
_MREMAP_MAYMOVE, _MREMAP_FIXED = 1, 2


def pinned_array(shape):
    """An FP64 numpy array in pinned host memory of exactly its size, which is given back when the array and all its
    views are gone; None where there is none to be had."""
    lib = nat.load()
    nbytes = 8 * int(np.prod(shape, dtype=np.int64))
    address = lib.lbm355_host_alloc(nbytes)
    if not address:
        return None
    _live[address] = nbytes
    memory = (ctypes.c_char * nbytes).from_address(address)
    weakref.finalize(memory, _give_back, lib, address).atexit = False
    return np.frombuffer(memory, dtype=np.float64).reshape(shape)


def _give_back(lib, address):
    if address in _inherited:
        _libc.munmap(address, _pages(_inherited.pop(address)))
        return
    _given_up.append(address)
    if torch.cuda.is_initialized() and torch.cuda.is_current_stream_capturing():
        return
    if _forking.acquire(blocking=False):
        try:
            while _given_up:
                address = _given_up.popleft()
                del _live[address]
                lib.lbm355_host_free(address)
        finally:
            _forking.release()


def _pages(nbytes):
    return -(-nbytes // mmap.PAGESIZE) * mmap.PAGESIZE


def _before_fork():
    _forking.acquire()
    for address, nbytes in list(_live.items()):
        copy = _libc.mmap(None, _pages(nbytes), mmap.PROT_READ | mmap.PROT_WRITE, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS,
                          -1, 0)
        if copy != _MAP_FAILED:
            ctypes.memmove(copy, address, nbytes)
            _copies.append((copy, address, nbytes))


def _after_fork_in_parent():
    for copy, _, nbytes in _copies:
        _libc.munmap(copy, _pages(nbytes))
    _copies.clear()
    _forking.release()


def _after_fork_in_child():
    for copy, address, nbytes in _copies:
        _libc.mremap(copy, _pages(nbytes), _pages(nbytes), _MREMAP_MAYMOVE | _MREMAP_FIXED, address)
        _inherited[address] = nbytes
    _copies.clear()
    _live.clear()
    _given_up.clear()
    _forking.release()


os.register_at_fork(before=_before_fork, after_in_parent=_after_fork_in_parent, after_in_child=_after_fork_in_child)
