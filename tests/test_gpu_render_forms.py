"""The render kernels' three forms (the reference's 32 x 32-thread blocks, two vote groups a
wave in 32 x 4-thread blocks, one in 32 x 8) give the same pixel records, bit for bit: images
whose edges cut the 8 x 4 vote groups and the blocks, down to one pixel, from few samples to
the most; main frames, and advanced ones that reuse, sample and foveate a zoomed-in frame's
pixels."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEAHORSE = (-0.743643887037151, 0.131825904205330)


class _Point(C.Structure):
    _fields_ = [("x", C.c_uint), ("y", C.c_uint)]


def _rect(real, centre, span, w, h):
    class Rect(C.Structure):
        _fields_ = [(n, real) for n in ("lbx", "lby", "rtx", "rty")]

    hw, hh = span / 2, span / 2 * h / w
    return Rect(centre[0] - hw, centre[1] - hh, centre[0] + hw, centre[1] + hh)


class _Forms:
    """Launches of a module's render kernels by name, without the renderer layer."""

    def __init__(self, cu, fractal, w, h):
        self.cu, self.w, self.h, self.L = cu, w, h, cu.abi.load()
        self.module = C.c_void_p()
        cu.abi.check(self.L.cu_module_load(f"{cu.KERNELS_DIR}/{fractal}.hsaco".encode(),
                                           C.byref(self.module)))
        self.planes = []
        for _ in range(2):
            p, pitch = C.c_void_p(), C.c_size_t()
            cu.abi.check(self.L.cu_mem_alloc_pitch(C.byref(p), C.byref(pitch), w * 16, h, 16))
            self.planes.append((p, pitch))

    def close(self):
        for p, _ in self.planes:
            self.cu.abi.check(self.L.cu_mem_free(p))
        self.cu.abi.check(self.L.cu_module_unload(self.module))

    def run(self, kernel, threads, pixel_rows, args, plane):
        """The records that `kernel` writes into `plane`, which is filled with 0xAA before."""
        check, (out, pitch) = self.cu.abi.check, self.planes[plane]
        mark = np.full(pitch.value * self.h, 0xAA, dtype=np.uint8)
        check(self.L.cu_memcpy_htod(out, mark.ctypes.data_as(C.c_void_p), mark.nbytes))
        fn = C.c_void_p()
        check(self.L.cu_module_get_function(self.module, kernel.encode(), C.byref(fn)))
        args = [C.c_void_p(out.value), C.c_long(pitch.value), _Point(self.w, self.h)] + args
        params = (C.c_void_p * len(args))(*[C.cast(C.pointer(a), C.c_void_p) for a in args])
        check(self.L.cu_launch_kernel(fn, (self.w + 31) // 32,
                                      (self.h + pixel_rows - 1) // pixel_rows, 1, 32, threads, 1, 0,
                                      params))
        check(self.L.cu_ctx_synchronize())
        got = np.zeros((self.h, self.w, 4), dtype=np.uint32)
        check(self.L.cu_memcpy_2d_dtoh(got.ctypes.data_as(C.c_void_p), self.w * 16, out,
                                       pitch.value, self.w * 16, self.h))
        return got


@pytest.mark.parametrize("size", [(1, 1), (8, 4), (33, 5), (39, 31), (100, 67)])
@pytest.mark.parametrize("precision,fractal,centre,span,limit", [
    (64, "mandelbrot", SEAHORSE, 1e-4, 3000), (32, "mandelbrot", (-0.5, 0.0), 3.0, 700),
    (32, "julia", (0.0, 0.0), 3.2, 400), (64, "mandelbrot", (-0.16, 1.04), 0.02, 13)])
def test_forms_agree(gpu, size, precision, fractal, centre, span, limit):
    cu, (w, h) = gpu, size
    real, word = (C.c_double, "Double") if precision == 64 else (C.c_float, "Float")
    forms = _Forms(cu, fractal, w, h)
    shapes = (("", 32, 32), ("Strip", 4, 4), ("Group", 8, 4))
    old, new = _rect(real, centre, span, w, h), _rect(real, centre, span * 0.93, w, h)
    try:
        for samples, flags in ((1.0, 0), (2.0, cu.FLAG_ADAPTIVE_SS), (5.0, cu.FLAG_ADAPTIVE_SS),
                               (7.0, 0), (64.0, cu.FLAG_ADAPTIVE_SS), (64.0, 0)):
            got = [forms.run("fractalRenderMain" + word + s, t, r,
                             [old, C.c_uint(limit), C.c_float(samples), C.c_uint(flags)], 0)
                   for s, t, r in shapes]
            assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
            advanced = (flags | cu.FLAG_SAMPLE_REUSE | cu.FLAG_FOVEATION | cu.FLAG_ZOOMING |
                        cu.FLAG_ZOOMING_IN)
            source, pitch = forms.planes[0]
            got = [forms.run("fractalRenderAdvanced" + word + s, t, r,
                             [new, C.c_uint(limit), C.c_float(samples), C.c_uint(advanced), old,
                              C.c_void_p(source.value), C.c_long(pitch.value), _Point(w // 2, h // 3)],
                             1)
                   for s, t, r in shapes]
            assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    finally:
        forms.close()
