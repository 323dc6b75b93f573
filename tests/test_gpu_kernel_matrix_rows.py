"""KernelMatrix rows written as whole lines: target counts around the columns
that one workgroup writes, row starts at every offset within a 128-byte line
(odd leading dimensions and an output that starts inside a line), and nothing
written outside the matrix, against the oracle.

Tolerance: 1e-13 normwise, the FP64 bar of the other tests.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [0, 1, 2, 4, 6, 9, 11])
@pytest.mark.parametrize("nt", [1, 15, 240, 241, 242, 251, 253, 509])
def test_rows(gpu, k, nt):
    rng = np.random.default_rng(100 * k + nt)
    _, K0, K1, _, _ = oracle.dims(k)
    for ns, shift in ((1, 0), (5, 3), (18, 13)):
        xt, xs = rng.random(3 * nt), rng.random(3 * ns)
        xt[:3] = xs[:3]
        n = rng.standard_normal(3 * ns)
        ref = oracle.kernel_matrix(k, xt, xs, n).ravel()
        size = ns * K0 * nt * K1
        d = [gpu.DeviceArray.from_host(a) for a in (xt, xs, n)]
        out = gpu.DeviceArray.from_host(np.full(size + 64, 7.5))
        gpu.check(gpu.lib().sctl_amd_kernel_matrix(k, -1, d[0].ptr, nt, d[1].ptr, d[2].ptr, ns,
                                                   ctypes.c_void_p(out.ptr.value + 8 * (16 + shift)), 0, None))
        gpu.synchronize()
        got = out.download()
        assert (got[:16 + shift] == 7.5).all() and (got[16 + shift + size:] == 7.5).all()
        assert np.abs(got[16 + shift:16 + shift + size] - ref).max() <= 1e-13 * np.abs(ref).max()
