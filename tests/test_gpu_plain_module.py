"""A module that exports the ABI's kernels and no others is launched in the reference's
geometry throughout, 32 x 32-thread blocks with one thread a pixel: every pixel of the
image is written, by the renderer layer and by the serving loop."""
import importlib
import os

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SIZES = [(2, 3), (33, 31), (64, 32), (100, 67)]


@pytest.fixture(scope="module")
def modules(gpu, tmp_path_factory):
    """A kernels directory whose mandelbrot module is tests/modules/plain_module.hip."""
    d = tmp_path_factory.mktemp("modules")
    os.symlink(os.path.join(ROOT, "tests", "modules", "mandelbrot.hsaco"), d / "mandelbrot.hsaco")
    os.symlink(os.path.join(gpu.KERNELS_DIR, "escape_family.hsaco"), d / "escape_family.hsaco")
    return str(d)


@pytest.mark.parametrize("w,h", SIZES)
def test_renderer_writes_every_pixel(gpu, modules, w, h):
    provider = gpu.FractalRendererProvider(modules)
    r = provider.get_renderer("mandelbrot")
    r.initialize_rendering(w, h, np.full(16, 1000, np.uint32))
    try:
        m = gpu.RenderingModel()
        m.set_segment(*gpu.plane_segment_from_center(-0.5, 0.0, 2.0, w, h))
        m.max_iterations, m.max_super_sampling = 100, 4.0
        for draw in (r.render_quality, r.render_fast):
            draw(m)
            assert np.array_equal(r.read_output().ravel(), 1000 + np.arange(w * h, dtype=np.uint32))
    finally:
        r.free_rendering_resources()
        provider.close()


@pytest.mark.parametrize("w,h", SIZES)
def test_server_writes_every_pixel(gpu, modules, w, h):
    serve = importlib.import_module("chaos-ultra_amd.serve")
    server = serve.Server(modules, 1 << 30)
    try:
        session = server.open(w, h, np.full(16, 1000, np.uint32))
        for tag in range(2):
            server.submit(session, (-0.5, 0.0), 2.0, 100, tag)
            done = []
            while not done:
                done = server.poll(10)
            assert done[0].status == 0, server.last_failure()
            assert np.array_equal(server.read_rgba(session, w, h).ravel(),
                                  1000 + np.arange(w * h, dtype=np.uint32))
    finally:
        server.close()
