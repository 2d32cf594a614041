"""The served frame's checksum, sum of rgba[i] * (2i + 1) mod 2^64, against numpy on
the image read back: sizes of four words, a few, no multiple of four, one block's
span and more than all blocks' first pass."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(2, 2), (3, 2), (5, 3), (32, 32), (37, 23), (1283, 7), (2047, 1029)])
def test_checksum_of_served_frame(gpu, w, h):
    sv = importlib.import_module("chaos-ultra_amd.serve")
    server = sv.Server(gpu.KERNELS_DIR, 1 << 30, slots=1)
    try:
        sid = server.open(w, h, gpu.default_palette())
        server.submit(sid, (-0.5, 0.1), 3.0, 64, 7)
        done = []
        while not done:
            done = server.poll(5)
        assert done[0].status == 0
        rgba = server.read_rgba(sid, w, h).ravel().astype(np.uint64)
        weight = 2 * np.arange(w * h, dtype=np.uint64) + np.uint64(1)
        assert done[0].checksum == int((rgba * weight).sum(dtype=np.uint64))
    finally:
        server.close()
