"""The persistent batch's queue: which items waves take without the counter, and that each
pixel is rendered once, in its own place, in whatever order and grabs the queue goes through
the tiles.  Oracle: every step of each orbit; counts and totals are whole numbers."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VIEWS = [dict(box=(-2.0, -1.25, 0.75, 1.25)), dict(box=(-1.80, -0.05, -1.72, 0.05)),
         dict(box=(-1.5, -1.5, 1.5, 1.5), kind=1, julia_c=(-0.12, 0.74))]


def batch_of(cu, tiles, precision=64):
    return importlib.import_module("chaos-ultra_amd.autotune").PersistentBatch(cu, tiles, precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,side,limit", [(16, 256, 50), (256, 64, 50), (1, 1024, 1000), (256, 16, 50)])
def test_shallow_batches_need_no_grabs(gpu, engine, n, side, limit, precision):
    """A batch that 4096 waves' first 256 items cover leaves the counter alone: each atomic
    on it takes 13 ns, and 64-item grabs took longer than the pixels."""
    batch = batch_of(gpu, [gpu.make_tile(-2, -1.5, 1, 1.5, side, side, limit)] * n, precision)
    batch.render(engine, gpu.Tune(32, 32, 256, 16))
    gpu.synchronize()
    assert batch.queue.download(np.uint64)[0] == 0


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("chunk", [1, 3, 64, 256])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 256, 257, 1024])
def test_every_pixel_once_in_depth_order(gpu, engine, oracle, n, chunk, precision):
    """Depths from the shallowest to past the one from which batches are always ordered,
    classes' edges among them; with a chunk of 1 or 3 the counter hands out most items."""
    rng = np.random.default_rng(n)
    limits = [1, 2, 3, 5, 6, 7, 8, 95, 96, 97, 127, 128, 4095, 4096, 5000, 6143, 6144, 8192]
    wide = 40 if n < 256 else 12
    tiles = []
    for _ in range(n):
        v = VIEWS[rng.integers(len(VIEWS))]
        tiles.append(gpu.make_tile(*v["box"], int(rng.integers(1, wide)), int(rng.integers(1, 7)),
                                   int(rng.choice(limits)), 4.0, kind=v.get("kind", 0),
                                   julia_c=v.get("julia_c", (0.0, 0.0))))
    tiles[n // 2].max_iter = 8192
    batch = batch_of(gpu, tiles, precision)
    batch.render(engine, gpu.Tune(16, 8, chunk, 16))
    gpu.synchronize()
    counts = batch.counts.download(np.uint32)
    total, offset = 0, 0
    for t in tiles:
        size = t.width * t.height
        want, _, steps = oracle.escape_tile(t, precision)
        assert np.array_equal(counts[offset:offset + size], want.ravel())
        total += steps
        offset += size
    assert batch.iters.total() == total
