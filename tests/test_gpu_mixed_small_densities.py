"""Mixed Evals of densities and normals near the lower end of FP32's range keep
their digits, though the matrix cores may flush what lies below 2^-126: every
kernel at a size above the one from which mixed precision runs its own kernels,
and the matrix-core kernels of three outputs at theirs, against the FP64 Eval of
the same densities.  1e-6 normwise, the mixed bar; down to where products of
densities and positions stay normal, sums scaled by a power of two are the same
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(k, 701, 300001) for k in range(16)] + [(2, 70001, 30001), (3, 40001, 30001), (4, 70001, 30001)]


@pytest.mark.parametrize("k,nt,ns", CASES, ids=["%d-%dx%d" % c for c in CASES])
def test_small(gpu, k, nt, ns):
    _, K0, K1, ND, _, _, _ = gpu.kernel_info(k)
    rng = np.random.default_rng(k)
    xt, xs, n, v = rng.random(3 * nt), rng.random(3 * ns), rng.standard_normal(3 * ns), rng.standard_normal(K0 * ns)
    d = [gpu.DeviceArray.from_host(a) for a in (xt, xs)]
    ctx = 3.0 if k >= 12 else None

    def run(prec, sn, sv):
        dn, dv = gpu.DeviceArray.from_host(n * sn), gpu.DeviceArray.from_host(v * sv)
        o = gpu.DeviceArray.from_host(np.zeros(nt * K1))
        gpu.eval(k, d[0], d[1], dn, dv, o, precision=prec, ctx=ctx)
        gpu.synchronize()
        return o.download()

    want, ordinary = run(gpu.FP64, 1.0, 1.0), run(gpu.MIXED, 1.0, 1.0)
    norm = np.linalg.norm(want)
    for sn, sv in [(1.0, 2.0 ** -110), (1.0, 2.0 ** -117)] + [(2.0 ** -117, 1.0), (2.0 ** -60, 2.0 ** -57)] * bool(ND):
        out = run(gpu.MIXED, sn, sv) / sn / sv
        assert np.linalg.norm(out - want) <= 1e-6 * norm, (sn, sv)
    assert np.linalg.norm(ordinary - want) <= 1e-6 * norm
    assert np.array_equal(run(gpu.MIXED, 1.0, 2.0 ** 20), ordinary * 2.0 ** 20)
    assert np.array_equal(run(gpu.MIXED, 1.0, 2.0 ** -60), ordinary * 2.0 ** -60)
    assert (run(gpu.MIXED, 1.0, 0.0) == 0).all()
