"""Reads of near lists into device memory: several threads read one list at
once, each on its own stream, the list is destroyed without waiting for them and
others of the same size are built and destroyed at once; every reader gets the
list's own results, bit for bit."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(seed, nelem, nt):
    rng = np.random.default_rng(seed)
    cnt = rng.integers(1, 130, nelem)
    dsp = np.concatenate(([0], np.cumsum(cnt)[:-1]))
    xs = np.repeat(rng.random((nelem, 3)), cnt, axis=0) + 0.02 * rng.standard_normal((cnt.sum(), 3))
    return rng.random(3 * nt), xs.ravel(), rng.uniform(0.01, 0.2, cnt.sum()), cnt, dsp


class Built:
    """A list built from device arrays."""

    def __init__(self, S, d, stream=None):
        self.S, self.nt, self.ne = S, d[0].shape[0] // 3, d[3].shape[0]
        self.h, n = ctypes.c_void_p(), ctypes.c_int64()
        S.check(S.lib().sctl_amd_near_list_build(ctypes.byref(self.h), d[0].ptr, self.nt, None, d[1].ptr,
                                                 d[1].shape[0] // 3, d[2].ptr, self.ne, d[3].ptr, d[4].ptr, 0, stream))
        S.check(S.lib().sctl_amd_near_list_size(self.h, ctypes.byref(n)))
        self.n = n.value

    def outputs(self):
        return [self.S.DeviceArray(3 * self.n)] + [self.S.DeviceArray(k, np.int64)
                                                   for k in (self.ne, self.ne, self.n, self.nt, self.nt)]

    def get(self, out, stream=None):
        p = [None if o is None else o.ptr for o in out]
        self.S.check(self.S.lib().sctl_amd_near_list_get(self.h, p[0], None, *p[1:], 0, stream))

    def destroy(self):
        self.S.check(self.S.lib().sctl_amd_near_list_destroy(self.h))


def arrays(S, c):
    return [S.DeviceArray.from_host(a, dtype=np.int64 if i > 2 else np.float64) for i, a in enumerate(c)]


KEYS = ("Xtrg_near", "near_elem_cnt", "near_elem_dsp", "near_scatter_index", "near_trg_cnt", "near_trg_dsp")


def streams(S, n):
    s = [ctypes.c_void_p() for _ in range(n)]
    for q in s:
        S.check(S.lib().sctl_amd_stream_create(ctypes.byref(q)))
    return s


def test_threads_read_one_list(gpu):
    c = case(1, 300, 40000)
    want = gpu.near_list(*c)
    d, other = arrays(gpu, c), arrays(gpu, case(2, 300, 40000))
    ss = streams(gpu, 4)
    with ThreadPoolExecutor(4) as pool:
        for _ in range(25):
            lst = Built(gpu, d)
            outs = [lst.outputs() for _ in ss]
            list(pool.map(lambda k: [lst.get(outs[k], ss[k]) for _ in range(3)], range(4)))
            lst.destroy()
            for _ in range(2):
                Built(gpu, other).destroy()
            for q in ss:
                gpu.synchronize(q)
            for out in outs:
                for key, o in zip(KEYS, out):
                    assert np.array_equal(o.download(), want[key]), key
    for q in ss:
        gpu.check(gpu.lib().sctl_amd_stream_destroy(q))


def test_some_outputs(gpu):
    c = case(3, 50, 3000)
    want = gpu.near_list(*c)
    lst = Built(gpu, arrays(gpu, c))
    for only in range(6):
        out = [o if i == only else None for i, o in enumerate(lst.outputs())]
        lst.get(out)
        gpu.synchronize()
        assert np.array_equal(out[only].download(), want[KEYS[only]])
    lst.get([None] * 6)
    lst.destroy()


def test_captured_read(gpu):
    """A read captured into a graph and replayed between eager reads; the list is destroyed with a launch under way
    and others are built at once."""
    hip = ctypes.CDLL("libamdhip64.so")

    def ok(status):
        assert status == 0

    c = case(4, 300, 40000)
    want = gpu.near_list(*c)
    d, other = arrays(gpu, c), arrays(gpu, case(5, 300, 40000))
    (q,) = streams(gpu, 1)
    for _ in range(5):
        lst = Built(gpu, d)
        out, eager = lst.outputs(), lst.outputs()
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        ok(hip.hipStreamBeginCapture(q, 2))  # relaxed
        lst.get(out, q)
        ok(hip.hipStreamEndCapture(q, ctypes.byref(graph)))
        ok(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)))
        for last in (False, False, True):
            for o in out:
                o.upload(np.full(o.shape, -1, o.dtype))
            ok(hip.hipGraphLaunch(run, q))
            if last:
                lst.destroy()
                for _ in range(2):
                    Built(gpu, other).destroy()
            else:
                lst.get(eager, q)
            gpu.synchronize(q)
            for key, o, e in zip(KEYS, out, eager):
                assert np.array_equal(o.download(), want[key]) and np.array_equal(e.download(), want[key]), key
        ok(hip.hipGraphExecDestroy(run))
        ok(hip.hipGraphDestroy(graph))
    gpu.check(gpu.lib().sctl_amd_stream_destroy(q))


def test_outputs_not_on_the_lists_gpu(gpu):
    """Outputs that are not memory of the list's GPU (one of them here: page-locked host memory) take the runtime's
    copies instead of the copy kernel."""
    hip = ctypes.CDLL("libamdhip64.so")
    c = case(6, 50, 3000)
    want = gpu.near_list(*c)
    lst = Built(gpu, arrays(gpu, c))
    out, p = lst.outputs(), ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(8 * lst.n), 0) == 0
    ptrs = [o.ptr for o in out]
    ptrs[3] = p
    gpu.check(gpu.lib().sctl_amd_near_list_get(lst.h, ptrs[0], None, *ptrs[1:], 0, None))
    gpu.synchronize()
    got = [o.download() for o in out]
    got[3] = np.array((ctypes.c_int64 * lst.n).from_address(p.value))
    for key, g in zip(KEYS, got):
        assert np.array_equal(g, want[key]), key
    lst.destroy()
    assert hip.hipHostFree(p) == 0
