"""Orbits that become cycles of states stop early in the kernels' unchecked blocks;
counts, smooth values and iteration totals stay those of the full loop, so each
engine is compared with the oracle (which runs every step) on views with much
interior, at iteration limits around the first held state, the block ends and the
first tests.  Counts and iterations are whole numbers and must be equal; smooth
values are within 1e-12 relative, as in the other kernel tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMOOTH_RTOL = 1e-12
# around kCycleFirst = 64, block ends, the first held states' tests, and far past them
LIMITS = [1, 63, 64, 65, 79, 80, 81, 97, 112, 113, 300, 3001]
VIEWS = {
    "home": dict(box=(-2.0, -1.25, 0.75, 1.25)),
    "period3": dict(box=(-1.80, -0.05, -1.72, 0.05)),
    "axis": dict(box=(-1.5, -0.01, 0.5, 0.01)),  # the real axis: y stays 0 at the middle row
    "julia_bounded": dict(box=(-1.5, -1.5, 1.5, 1.5), kind=1, julia_c=(-0.12, 0.74)),
    "julia_zero": dict(box=(-1.25, -1.25, 1.25, 1.25), kind=1, julia_c=(0.0, 0.0)),
}


def tile_of(cu, view, limit, spp, bailout=4.0, size=(53, 37)):
    v = VIEWS[view]
    return cu.make_tile(*v["box"], *size, limit, bailout, kind=v.get("kind", 0),
                        julia_c=v.get("julia_c", (0.0, 0.0)), spp=spp,
                        pattern=cu.SAMPLE_JITTER if spp > 1 else cu.SAMPLE_CENTRE, seed=limit)


def same(got, want):
    (c, s, it), (wc, ws, wit) = got, want
    assert np.array_equal(c.reshape(wc.shape), wc)
    assert it == wit
    rel = np.abs(s.reshape(ws.shape) - ws) / np.maximum(np.abs(ws), 1.0)
    assert rel.max() <= SMOOTH_RTOL


def grid(cu, engine, tile, precision):
    n = tile.width * tile.height
    counts, smooth, iters = cu.DeviceBuffer(n * 4), cu.DeviceBuffer(n * 8), cu.IterationCounter()
    engine.escape_tile(precision, tile, counts, smooth, iters)
    cu.synchronize()
    return counts.download(np.uint32), smooth.download(np.float64), iters.total()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("spp", [1, 3])
@pytest.mark.parametrize("view", sorted(VIEWS))
def test_grid_kernel(gpu, engine, oracle, view, spp, precision):
    for limit in LIMITS:
        tile = tile_of(gpu, view, limit, spp)
        same(grid(gpu, engine, tile, precision), oracle.escape_tile(tile, precision))


def deep_case(cu, engine, oracle, desc, method):
    """A deep frame and the oracle's checked loop over its pixels, bit for bit."""
    f = cu.DeepFrame(engine, desc, method)
    f.render()
    rep, counts = f.report(), f.counts()
    orbit = f.orbit() if method != cu.DEEP_DIRECT_F64 else None
    f.close()
    ys, xs = np.mgrid[0:desc.height, 0:desc.width]
    om = {cu.DEEP_DIRECT_F64: oracle.DEEP_DIRECT_F64, cu.DEEP_PERTURB_F32: oracle.DEEP_PERTURB_F32,
          cu.DEEP_PERTURB_F64: oracle.DEEP_PERTURB_F64}[method]
    wc, _, _, wit = oracle.deep_pixels(om, xs.ravel(), ys.ravel(), desc, orbit, rep.reference_length)
    assert np.array_equal(counts.ravel(), wc)
    assert rep.iterations == wit


@pytest.mark.parametrize("limit", LIMITS)
def test_direct_deep_frame(gpu, engine, oracle, limit):
    deep_case(gpu, engine, oracle, gpu.make_deep(-0.25, 0.125, 1.5, 61, 39, limit, 16.0),
              gpu.DEEP_DIRECT_F64)


# (centre, height of the view, precision): the whole set in FP32; FP64 views below the
# float ulp inside the period-2 disk's edge and inside the period-3 island
RENDER_VIEWS = [("mandelbrot", (-0.5, 0.0), 2.5, 32), ("mandelbrot", (-1.25, 0.0), 2e-6, 64),
                ("mandelbrot", (-1.7548777, 0.0), 2e-6, 64), ("julia", (0.0, 0.0), 3.0, 32)]


@pytest.mark.parametrize("fractal,centre,zoom,precision", RENDER_VIEWS)
@pytest.mark.parametrize("samples,adaptive", [(1.0, 0), (4.0, 0), (5.0, 1)])
def test_module_kernels(gpu, oracle, fractal, centre, zoom, precision, samples, adaptive):
    """The main kernel's pooled orbits (first held state at 128), FP32 and FP64."""
    cu, w, h = gpu, 67, 45
    provider = cu.FractalRendererProvider()
    r = provider.get_renderer(fractal)
    kind, jc = (cu.FRACTAL_JULIA, (-0.12, 0.74)) if fractal == "julia" else (cu.FRACTAL_MANDELBROT, (0, 0))
    if fractal == "julia":
        r.set_fractal_custom_params("-0.12;0.74")
    r.initialize_rendering(w, h, cu.default_palette())
    try:
        seg = cu.plane_segment_from_center(*centre, zoom, w, h)
        for limit in LIMITS + [127, 128, 129, 144, 145, 192, 208]:
            m = cu.RenderingModel()
            m.set_segment(*seg)
            m.max_iterations, m.max_super_sampling = limit, samples
            m.use_adaptive_super_sampling = adaptive
            before = r.iterations()
            r.render_quality(m)
            oracle.render_iterations()
            want = oracle.render_main(precision, kind, jc, w, h, seg, limit, samples,
                                      cu.FLAG_ADAPTIVE_SS if adaptive else 0)
            assert r.iterations() - before == oracle.render_iterations()
            got = r.read_pixel_info()
            for field in ("value", "weight", "is_reused", "weight_of_new_samples"):
                assert np.array_equal(got[field], want[field]), (limit, field)
    finally:
        r.free_rendering_resources()
        provider.close()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("spp", [1, 3])
@pytest.mark.parametrize("steps,chunk,refill", [(8, 64, 1), (16, 256, 16), (32, 100, 64)])
def test_persistent_kernel(gpu, engine, oracle, steps, chunk, refill, spp, precision):
    """All views and limits (and one bailout below 4, which takes checked steps) as one batch."""
    import importlib
    at = importlib.import_module("chaos-ultra_amd.autotune")
    limits = LIMITS + [7, 8, 15, 16, 31, 32, 33, 128, 159, 160, 161]
    tiles = [tile_of(gpu, v, n, spp, size=(29, 17)) for v in sorted(VIEWS) for n in limits]
    tiles.append(tile_of(gpu, "home", 300, spp, bailout=3.0))
    batch = at.PersistentBatch(gpu, tiles, precision)
    batch.render(engine, gpu.Tune(steps, 8, chunk, refill))
    gpu.synchronize()
    counts, smooth = batch.counts.download(np.uint32), batch.smooth.download(np.float64)
    total, offset = 0, 0
    for t in tiles:
        n = t.width * t.height
        wc, ws, wit = oracle.escape_tile(t, precision)
        same((counts[offset:offset + n], smooth[offset:offset + n], wit), (wc, ws, wit))
        total += wit
        offset += n
    assert batch.iters.total() == total


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("spp", [1, 4])
@pytest.mark.parametrize("tune", [(16, 24, 0, 0, 40), (8, 32, 3, 1, 0), (16, 1, 1, 2, 64), (8, 16, 2, 0, 1)])
def test_frame_pipeline(gpu, engine, oracle, tune, spp, precision):
    """All views and limits as the tiles of one frame: pass 1, tail passes and drain."""
    limits = LIMITS + [7, 8, 15, 16, 17, 128, 143, 144, 145, 192, 193]
    tiles = [tile_of(gpu, v, n, spp, size=(29, 17)) for v in sorted(VIEWS) for n in limits]
    tiles.append(tile_of(gpu, "home", 300, spp, bailout=3.0))
    frame = gpu.Frame(engine, tiles, precision)
    frame.render(gpu.FrameTune(*tune))
    gpu.synchronize()
    counts, smooth = frame.counts(), frame.smooth()
    total, offset = 0, 0
    for t in tiles:
        n = t.width * t.height
        wc, ws, wit = oracle.escape_tile(t, precision)
        same((counts[offset:offset + n], smooth[offset:offset + n], wit), (wc, ws, wit))
        total += wit
        offset += n
    assert frame.iterations() == total
    frame.close()


# (centre, width, limit): a reference that escapes early so that every interior pixel
# rebases, one inside the set, one of a few steps (checked steps only), a shallow frame
@pytest.mark.parametrize("centre,width,limit", [
    ((-0.743643887037151, 0.131825904205330), 1e-6, 30000),
    ((-0.743643887037151 + 4e-8, 0.131825904205330 - 6e-8), 1e-6, 30000),
    ((0.5, 0.0), 1e-3, 3000), ((0.26, 1e-3), 0.05, 4000), ((-0.25, 0.125), 1.0, 2000),
    ((-1.0, 0.0), 0.5, 700), ((0.0, 0.0), 0.5, 97)])
@pytest.mark.parametrize("method", [32, 64])
def test_perturbation(gpu, engine, oracle, centre, width, limit, method):
    """Rebased deltas that come back end the pixel with the checked loop's result."""
    deep_case(gpu, engine, oracle, gpu.make_deep(*centre, width, 45, 27, limit, 256.0), method)


# references that settle into cycles of 1, 2, 3, 4, 10 and 78 entries, at different rates; the
# limits are no multiples of a block's 32 steps, and the second frame keeps the first's orbit
@pytest.mark.parametrize("centre,width", [
    ((-0.4, 0.05), 0.9), ((-1.02, 0.03), 0.3), ((-0.123, 0.745), 0.12),
    ((0.2823, 0.5301), 0.05), ((-0.5355, 0.6085), 0.02), ((-0.7436440753, 0.1318253789), 1e-6)])
@pytest.mark.parametrize("method", [32, 64])
def test_perturbation_along_a_periodic_reference(gpu, engine, oracle, centre, width, method):
    """A delta that comes back a whole number of the reference's periods later ends the pixel
    with the checked loop's result, also with an orbit longer than the frame's limit."""
    om = oracle.DEEP_PERTURB_F32 if method == 32 else oracle.DEEP_PERTURB_F64
    desc = gpu.make_deep(*centre, width, 45, 27, 9001, 256.0)
    desc.flags |= gpu.abi.DEEP_REUSE_ORBIT
    frame = gpu.DeepFrame(engine, desc, method)
    ys, xs = np.mgrid[0:desc.height, 0:desc.width]
    for limit in (9001, 2999):
        desc.max_iter = limit
        frame.retarget(desc)
        frame.render()
        report = frame.report()
        assert report.references == (1 if limit == 9001 else 0)
        orbit = frame.orbit() if limit == 9001 else orbit
        wc, _, _, wit = oracle.deep_pixels(om, xs.ravel(), ys.ravel(), desc, orbit,
                                           report.reference_length)
        assert np.array_equal(frame.counts().ravel(), wc)
        assert report.iterations == wit
    frame.close()


# frames whose deltas grow from far below the reference's values to rebases and escapes, so that
# their blocks run without tests, then with them; the reference of the second comes close to 0
# every third step, the fourth's limit ends inside the first phase
@pytest.mark.parametrize("centre,width,limit", [
    ((-0.743643887037151, 0.131825904205330), 1e-12, 4001),
    ((-1.7548776662466927, 0.0), 1e-3, 1501), ((-1.7548776662466927, 1e-9), 1e-9, 1501),
    ((-0.743643887037151, 0.131825904205330), 1e-25, 1000), ((0.0, 1.0), 1e-10, 700),
    ((0.2501, 0.0), 1e-5, 999)])
@pytest.mark.parametrize("method", [32, 64])
def test_perturbation_blocks_without_tests(gpu, engine, oracle, centre, width, limit, method):
    """Blocks in which no rebase test can fire leave them out, with the checked loop's result."""
    deep_case(gpu, engine, oracle, gpu.make_deep(*centre, width, 45, 27, limit, 256.0), method)


# a batch's queue order: by depth up to 256 tiles, above as they come; ties, one pixel, tiles of a row
@pytest.mark.parametrize("n", [1, 2, 3, 64, 255, 256, 257, 700])
def test_persistent_kernel_order_of_tiles(gpu, engine, oracle, n):
    """Every tile's pixels land in its own place, whatever the order the queue takes them in."""
    import importlib
    at = importlib.import_module("chaos-ultra_amd.autotune")
    rng = np.random.default_rng(n)
    views = sorted(VIEWS)
    tiles = [tile_of(gpu, views[rng.integers(len(views))], int(rng.choice([1, 40, 40, 333, 700, 701])),
                     1, size=(int(rng.integers(1, 14)), int(rng.integers(1, 7)))) for _ in range(n)]
    batch = at.PersistentBatch(gpu, tiles, 64)
    batch.render(engine, gpu.Tune(16, 8, 64, 16))
    gpu.synchronize()
    counts, smooth = batch.counts.download(np.uint32), batch.smooth.download(np.float64)
    total, offset = 0, 0
    for t in tiles:
        m = t.width * t.height
        wc, ws, wit = oracle.escape_tile(t, 64)
        same((counts[offset:offset + m], smooth[offset:offset + m], wit), (wc, ws, wit))
        total += wit
        offset += m
    assert batch.iters.total() == total
