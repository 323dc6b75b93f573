"""A change of a plan's shape that finds no device memory is an error and leaves
the plan as it was: applies give what they gave, and the change can be made
later.  The partial sums of the cut blocks (28 MB) are what does not fit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_set_shape_without_memory(gpu):
    hip = ctypes.CDLL("libamdhip64.so")
    nb, nt, ns = 64, 128, 100000
    rng = np.random.default_rng(0)
    plan = gpu.Plan(3, np.arange(nb) * nt, np.full(nb, nt), np.zeros(nb), np.full(nb, ns), nb * nt, ns)
    plan.set_geometry(rng.random(3 * nb * nt), rng.random(3 * ns), rng.standard_normal(3 * ns))
    plan.set_shape(2, 2, 0)
    f = gpu.DeviceArray.from_host(rng.standard_normal(3 * ns))
    out = [gpu.DeviceArray.from_host(np.zeros(3 * nb * nt)) for _ in range(3)]
    plan.apply(f, out[0])
    gpu.synchronize()
    want, fill, have, total = out[0].download(), [], ctypes.c_size_t(), ctypes.c_size_t()
    with pytest.raises(gpu.SctlAmdError):
        gpu.DeviceArray(1 << 48, np.uint8)  # so that no memory is kept for near lists, which would be given up below
    assert hip.hipMemGetInfo(ctypes.byref(have), ctypes.byref(total)) == 0
    size = have.value
    while size >= 1 << 21:
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
            fill.append(p)
        else:
            size //= 2
    hip.hipGetLastError()  # the failed attempts'
    try:
        with pytest.raises(gpu.SctlAmdError) as e:
            plan.set_shape(2, 1, 0)
        assert e.value.status == 5  # SCTL_AMD_ERROR_OUT_OF_MEMORY
        plan.set_shape(2, 2, 0)
        assert plan.shape() == (2, 2, 0)
        plan.apply(f, out[1])
        gpu.synchronize()
    finally:
        for p in fill:
            assert hip.hipFree(p) == 0
    assert np.array_equal(out[1].download(), want)
    plan.set_shape(2, 1, 0)
    plan.apply(f, out[2])
    gpu.synchronize()
    assert np.abs(out[2].download() - want).max() <= 1e-13 * np.abs(want).max()
