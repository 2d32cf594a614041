"""Arrays read back from the device: each owns its values while it or a view of it is
alive, blocks are used again after that, and what is kept and lent is bounded."""
import gc
import importlib
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words", [1, 1000, (64 << 10) // 4 - 1, (64 << 10) // 4, 100003, 3 << 20])
def test_arrays_are_independent(gpu, words):
    a = np.arange(words, dtype=np.uint32)
    buf = gpu.DeviceBuffer.from_array(a)
    first = buf.download(np.uint32)
    view = first[::3].reshape(-1, 1)
    buf.upload(a + 7)
    second = buf.download(np.uint32)
    del first
    gc.collect()
    third = buf.download(np.uint32)
    second[0] = 0  # writable
    assert np.array_equal(view[:, 0], a[::3])
    assert np.array_equal(third, a + 7)


def test_blocks_are_bounded_and_shared_between_threads(gpu, monkeypatch):
    pkg = importlib.import_module("chaos-ultra_amd")
    pool = pkg._ReadBack()
    monkeypatch.setattr(pool, "CACHED", 1 << 20)
    monkeypatch.setattr(pool, "LENT", 4 << 20)
    kept = [pool.empty(1 << 18, np.uint32) for _ in range(6)]  # 1 MiB each: the last two are ordinary
    assert pool._lent == 4 << 20 and pool._cached == 0
    assert len({k.ctypes.data for k in kept}) == 6
    del kept
    gc.collect()
    assert pool._lent == 0 and 0 < pool._cached <= 1 << 20

    def work(seed):
        for k in range(50):
            x = pool.empty(50000 + 1000 * (k % 5), np.float64)
            x[:] = seed
            assert (x == seed).all()
    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gc.collect()
    assert pool._lent == 0 and pool._cached <= 1 << 20
