"""What the reference orbit's kernels leave in device memory for the pixel kernels: the
entries (equal to the oracle's), the cycle that they end in and each block's bound (equal to
plain restatements: whole numbers, and FP32 operations that round correctly on both sides)."""
import ctypes as C

import numpy as np
import pytest

from test_perturb_quiet_bound import STEPS, quiet_bounds

pytestmark = pytest.mark.gpu

PERIOD_MAX = 4096


def cycle(z, last, max_iter):
    """(period, start) of the entries' cycle; (0, 0) where the orbit escapes or none is found."""
    if last != max_iter or last == 0:
        return 0, 0
    same = np.nonzero((z[:last, :3] == z[last, :3]).all(1))[0]
    if same.size == 0 or last - same[-1] > PERIOD_MAX:
        return 0, 0
    period = last - same[-1]
    differ = np.nonzero((z[: last + 1 - period, :3] != z[period:, :3]).any(1))[0]
    return period, (differ[-1] + 1 if differ.size else 0)


# centre, limit, and the period that the view has been chosen for (None: it escapes)
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("centre,max_iter,period", [
    ((-0.4, 0.05), 9001, 1), ((-1.02, 0.03), 9001, 2), ((-0.123, 0.745), 9000, 3), ((0.2823, 0.5301), 9001, 4),
    ((-0.5355, 0.6085), 9001, 10), ((-0.7436440753, 0.1318253789), 9001, 78),
    ((-0.743643887037151, 0.131825904205330), 50000, None), ((0.5, 0.5), 64, None), ((0.0, 0.0), 32, 1),
    ((-0.4, 0.05), 1, None), ((-1.0, 0.0), 2, 2)])
def test_entries_cycle_and_bounds(gpu, oracle, centre, max_iter, period, precision):
    cu, L = gpu, gpu.abi.load()
    check = cu.abi.check
    real = np.float32 if precision == 32 else np.float64
    want, last = oracle.reference_orbit(*centre, max_iter, 256.0, precision)
    module, fn = C.c_void_p(), C.c_void_p()
    check(L.cu_module_load(f"{cu.KERNELS_DIR}/escape_family.hsaco".encode(), C.byref(module)))
    try:
        name = b"referenceOrbitFloat" if precision == 32 else b"referenceOrbitDouble"
        check(L.cu_module_get_function(module, name, C.byref(fn)))
        orbit = cu.DeviceBuffer(4 * real().nbytes * (max_iter + 1))
        info = cu.DeviceBuffer(16)
        args = [C.c_double(centre[0]), C.c_double(0), C.c_double(centre[1]), C.c_double(0), C.c_uint(max_iter),
                C.c_double(256.0), C.c_void_p(orbit.address), C.c_void_p(info.address)]
        params = (C.c_void_p * len(args))(*[C.cast(C.pointer(a), C.c_void_p) for a in args])
        check(L.cu_launch_kernel(fn, 1, 1, 1, 64, 1, 1, 0, params))
        check(L.cu_ctx_synchronize())
        got_last, got_period, got_start, _ = info.download(np.uint32)
        entries = orbit.download(real)[: 4 * (last + 1)].reshape(-1, 4)
    finally:
        check(L.cu_module_unload(module))
    assert got_last == last
    assert np.array_equal(entries[:, :3], want[:, :3])
    assert (got_period, got_start) == cycle(want, last, max_iter)
    if period is not None:
        assert got_period == period and got_start < max(max_iter // 4, 1)
    starts = np.arange(0, last // STEPS * STEPS, STEPS)
    bounds = np.zeros(last + 1, np.float32)
    bounds[starts] = quiet_bounds(want, starts) if starts.size else 0
    assert np.array_equal(entries[:, 3], bounds.astype(real))
