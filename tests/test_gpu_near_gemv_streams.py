"""One plan's near-field GEMV for two density vectors on two streams at once: a
call keeps nothing in the plan, so each result equals, bit for bit, the one
that the call gives alone.  Few blocks with long rows, so that rows are cut into
pieces: up to four of them (workgroups of four waves), more (of sixteen), none
beside some, a block without a matrix and one without sources; against the
oracle's product in 64 bits (1e-13 of the sum of magnitudes, FP64 sums of at
most 40 000 terms)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {"uncut": ([40, 3], [300, 511]),
         "four": ([17, 9, 8, 1, 5], [1500, 700, 2048, 64, 0]),
         "sixteen": ([9, 70, 3], [40001, 5, 9000])}


@pytest.mark.parametrize("name", sorted(CASES))
def test_two_streams_of_one_plan(gpu, name):
    tc, sc = (np.array(a) for a in CASES[name])
    td, sd = (np.concatenate(([0], np.cumsum(a)[:-1])) for a in (tc, sc))
    rng = np.random.default_rng(len(name))
    plan = gpu.Plan(0, td, tc, sd, sc, int(tc.sum()), int(sc.sum()))
    size = tc * sc
    off = np.concatenate(([0], np.cumsum(size)[:-1]))
    off[1] = -1
    n = plan.near_layout(off)
    Kh = rng.standard_normal(n)
    K = gpu.DeviceArray.from_host(Kh)
    Fh = [rng.standard_normal(sc.sum()) for _ in range(2)]
    F = [gpu.DeviceArray.from_host(f) for f in Fh]
    U = [gpu.DeviceArray.from_host(np.full(tc.sum(), 7.0)) for _ in range(2)]
    want = []
    for f, u in zip(F, U):
        plan.near_gemv(K, f, u)
        gpu.synchronize()
        want.append(u.download())
    for f, w in zip(Fh, want):
        for b in range(tc.size):
            got = w[td[b]:td[b] + tc[b]]
            if off[b] < 0 or sc[b] == 0:
                assert (got == 0).all()
                continue
            M, x = Kh[off[b]:off[b] + size[b]].reshape(tc[b], sc[b]), f[sd[b]:sd[b] + sc[b]]
            assert np.abs(got - M @ x).max() <= 1e-13 * (np.abs(M) @ np.abs(x)).max()
    s = [ctypes.c_void_p() for _ in range(2)]
    for q in s:
        gpu.check(gpu.lib().sctl_amd_stream_create(ctypes.byref(q)))
    for _ in range(40):
        for u in U:
            u.upload(np.full(tc.sum(), 7.0))
        for _ in range(8):
            for f, u, q in zip(F, U, s):
                plan.near_gemv(K, f, u, stream=q)
        for q in s:
            gpu.synchronize(q)
        for u, w in zip(U, want):
            assert np.array_equal(u.download(), w)
    for q in s:
        gpu.check(gpu.lib().sctl_amd_stream_destroy(q))
