"""A near list of few pairs and many targets with little device memory free: a
build's scratch follows what the list holds, not a fixed number of pairs per
target.  30 000 000 targets, 1200 of them near the elements; 64-bit pair keys.
In 5 GB the usual reserves fit; in 2.4 GB they
leave too little for the results and in 2 GB they do not fit, and the build goes
on with the sizes that it has counted."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

NT, NEAR, NELEM = 30_000_000, 1200, 200


def fill_but(hip, free):
    """Takes the device's memory but for `free` bytes; returns the blocks."""
    have, total, hold, fill = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_void_p(), []
    assert hip.hipMemGetInfo(ctypes.byref(have), ctypes.byref(total)) == 0
    if free:
        assert hip.hipMalloc(ctypes.byref(hold), ctypes.c_size_t(int(free))) == 0
    size = have.value
    while size >= 1 << 24:  # the rest, in blocks of halving size
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
            fill.append(p)
        else:
            size //= 2
    hip.hipGetLastError()  # the failed attempts'
    if free:
        assert hip.hipFree(hold) == 0
    return fill


@pytest.mark.parametrize("free", [2.0e9, 2.4e9, 5.0e9])
def test_little_memory(gpu, free):
    hip = ctypes.CDLL("libamdhip64.so")
    rng = np.random.default_rng(1)
    xt = 2.0 + rng.random((NT, 3))
    at = np.sort(rng.choice(NT, NEAR, replace=False))
    xt[at] = 0.8 * rng.random((NEAR, 3))
    xs, rad = 0.8 * rng.random((NELEM, 3)), rng.uniform(0.02, 0.2, NELEM)
    cnt, dsp = np.ones(NELEM, dtype=np.int64), np.arange(NELEM)
    want = oracle.default().near_list(xt[at].ravel(), xs.ravel(), rad, cnt, dsp)
    d = [gpu.DeviceArray.from_host(a.ravel()) for a in (xt, xs, rad)]
    d += [gpu.DeviceArray.from_host(a, dtype=np.int64) for a in (cnt, dsp)]
    gpu.synchronize()
    fill = fill_but(hip, free)
    try:
        got = gpu.near_list(*d)
    finally:
        for p in fill:
            assert hip.hipFree(p) == 0
    assert want["near_scatter_index"].size > 0
    for key in ("Xtrg_near", "near_elem_cnt", "near_elem_dsp", "near_scatter_index"):
        assert np.array_equal(got[key], want[key]), key
    for key in ("near_trg_cnt", "near_trg_dsp"):
        assert np.array_equal(got[key][at], want[key]), key
        assert np.count_nonzero(got[key]) == np.count_nonzero(want[key]), key


def test_kept_memory_goes_to_other_allocations(gpu):
    """The blocks kept between builds, more than a gigabyte here, are freed when another allocation fails."""
    hip = ctypes.CDLL("libamdhip64.so")
    rng = np.random.default_rng(2)
    d = [gpu.DeviceArray.from_host(a) for a in (2.0 + rng.random(3 * NT), rng.random(3), np.array([0.1]))]
    d += [gpu.DeviceArray.from_host(np.array([a]), dtype=np.int64) for a in (1, 0)]
    assert gpu.near_list(*d)["near_scatter_index"].size == 0
    fill = fill_but(hip, 0)
    try:
        a = gpu.DeviceArray(1 << 30, np.uint8)
        a.free()
    finally:
        for p in fill:
            assert hip.hipFree(p) == 0
