"""Arrays read back from the device, with the copies and the page-locked allocation
replaced by host stand-ins: which entry points return arrays that own their memory, and
what a forked child finds in arrays that do not."""
import ctypes as C
import gc
import importlib
import mmap
import os

import numpy as np
import pytest


@pytest.fixture
def pkg(monkeypatch):
    """The package with cu_host_alloc, cu_host_free and cu_memcpy_dtoh (which fills with
    0x01 bytes) on the host.  Blocks are shared mappings that a child does not get, as the
    driver's are (VmFlags "sh" and "dc")."""
    pkg = importlib.import_module("chaos-ultra_amd")
    blocks = {}

    def call(name, *args):
        if name == "cu_host_alloc":
            m = mmap.mmap(-1, args[1].value)
            m.madvise(mmap.MADV_DONTFORK)
            address = C.addressof(C.c_char.from_buffer(m))
            blocks[address] = m
            C.cast(args[0], C.POINTER(C.c_void_p))[0] = address
        elif name == "cu_host_free":
            del blocks[args[0].value]
        else:
            assert name == "cu_memcpy_dtoh"
            C.memset(args[0], 1, args[2].value)

    monkeypatch.setattr(pkg.abi, "call", call)
    monkeypatch.setattr(pkg, "_read_back", pkg._ReadBack())
    return pkg


def made(cls, **fields):
    thing = cls.__new__(cls)
    thing.__dict__.update(fields)
    return thing


@pytest.mark.parametrize("words", [0, 100, 100_000, 2_000_000])
def test_flat_arrays_own_their_memory(pkg, words):
    """They can be resized in place, as any array that numpy allocated."""
    buffer = made(pkg.DeviceBuffer, nbytes=4 * words, ptr=C.c_void_p())
    frame = made(pkg.Frame, total_pixels=words, d_counts=0, d_smooth=0, handle=None)
    for a in (buffer.download(np.uint32), buffer.download(np.uint8, 3 * words), frame.counts(),
              frame.smooth()):
        assert a.flags.owndata and a.flags.writeable and (a.view(np.uint8) == 1).all()
        a.resize(a.size + 5, refcheck=False)
        assert not a[-5:].any()


@pytest.mark.parametrize("kilobytes,locked", [(64, False), (383, False), (384, True), (8100, True)])
def test_small_images_are_ordinary_arrays(pkg, kilobytes, locked):
    """Page-locking a block for an image that is kept only pays from 384 KB on."""
    image = pkg._read_back.empty(256 * kilobytes, np.uint32)
    assert image.flags.owndata != locked
    assert (pkg._read_back._lent > 0) == locked


def in_child(work) -> int:
    """work() in a forked child: its exit status (the signal's number, negative, if it was
    killed), 0 if it returned true."""
    pid = os.fork()
    if pid == 0:
        status = 1
        try:
            status = 0 if work() else 1
        finally:
            os._exit(status)
    status = os.waitpid(pid, 0)[1]
    return -os.WTERMSIG(status) if os.WIFSIGNALED(status) else os.WEXITSTATUS(status)


def test_forked_child_has_its_own_arrays(pkg):
    """A child reads the values of the time of the fork, whatever either side writes or
    drops afterwards; the parent's arrays and blocks are as they were."""
    pool = pkg._read_back
    images = [pool.empty(n, np.uint32) for n in (200_000, 2_073_600, 300_001)]
    for k, a in enumerate(images):
        a[:] = np.arange(a.size, dtype=np.uint32) + k
    waiting = pool.empty(400_000, np.uint32)
    del waiting
    gc.collect()
    lent, cached, lock = pool._lent, pool._cached, pool._lock

    def child():
        ok = all(np.array_equal(a, np.arange(a.size, dtype=np.uint32) + k) for k, a in enumerate(images))
        for a in images:
            a[:] = 0
        del a
        images.clear()
        gc.collect()
        return ok and pool._lent == 0 and pool._cached == 0 and not pool._free

    assert in_child(child) == 0
    assert (pool._lent, pool._cached, pool._lock) == (lent, cached, lock) and not pool._copies
    for k, a in enumerate(images):
        assert np.array_equal(a, np.arange(a.size, dtype=np.uint32) + k)
    del a
    images.clear()
    gc.collect()
    assert pool._lent == 0 and pool._cached > cached
    assert in_child(lambda: pool._cached == 0) == 0
