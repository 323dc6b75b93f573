"""Mixed precision on both sides of the size from which it runs its own kernels,
with coincident points, flat and one-point sets, through sctl_amd_eval, a dense
plan (equal bit for bit) and sctl_amd_eval_noalloc, against the oracle.

Tolerance: 1e-6 of the largest sum of term magnitudes per target, the bound of
the mixed path for sums that cancel (each FP32 pair is good to a few 2^-24 of
itself); above it the sizes are ragged in targets, tiles and 64-source parts.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(13001, 12000), (1201, 130001), (140001, 1100)]


def sets(rng, where, nt, ns):
    xs, xt = rng.random((ns, 3)), rng.random((nt, 3))
    if where == "plane":
        xs[:, 2] = xt[:, 2] = 0.25
    elif where == "far":
        xt = xt * 0.1 + np.array([50.0, -20.0, 10.0])
    elif where == "point":
        xs[:] = xs[0]
        xt[: nt // 2] = xs[0]
    elif where == "tiny":  # |t'|^2 around 2^-100; the closest pairs' r^2 still normal in FP32
        xs, xt = xs * 1e-15, xt * 1e-15
    xt[:37] = xs[ns - 37:]
    return xt.ravel(), xs.ravel()


def magnitude(k, xt, xs, n, v):
    """Largest sum of |term| over the targets (Laplace kernels), on a subset of 64 targets."""
    t = xt.reshape(-1, 3)[:: max(1, xt.size // 192)][:64]
    d = t[:, None, :] - xs.reshape(-1, 3)[None]
    r2 = (d * d).sum(-1)
    with np.errstate(divide="ignore", invalid="ignore"):
        z = np.where(r2 > 0, 1 / np.sqrt(r2), 0.0)
    w = np.abs(v)[None] * z if k == 0 else np.abs((d * n.reshape(-1, 3)[None]).sum(-1) * v[None]) * z ** 3
    return (w.sum(1) / (4 * np.pi)).max()


@pytest.mark.parametrize("where", ["cube", "plane", "far", "point", "tiny"])
@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d" % s for s in SHAPES])
@pytest.mark.parametrize("k", [0, 1])
def test_both_sides(gpu, k, shape, where):
    if where == "tiny" and k == 1:
        pytest.skip("r^-3 leaves FP32's range there, in this path as in any FP32 one")
    nt, ns = shape
    rng = np.random.default_rng(nt + k)
    xt, xs = sets(rng, where, nt, ns)
    n, v = rng.standard_normal(3 * ns), rng.uniform(-1, 1, ns)
    for m in (ns, 1.4e8 / nt):  # its own kernels; the FP64 kernels
        m = min(ns, int(m))
        a = (xt, xs[3 * (ns - m):], n[3 * (ns - m):], v[ns - m:])
        ref = oracle.eval(k, *a)
        out = gpu.eval(k, *a, precision=gpu.MIXED)
        bar = 1e-6 * max(np.abs(ref).max(), magnitude(k, *a))
        assert np.isfinite(out).all()
        assert np.abs(out - ref).max() <= bar
        plan = gpu.DensePlan(k, *a[:3], precision=gpu.MIXED)
        assert np.array_equal(plan.apply(a[3]), out)
        d = [gpu.DeviceArray.from_host(q) for q in a]
        o = gpu.DeviceArray.from_host(np.zeros(nt))
        gpu.check(gpu.lib().sctl_amd_eval_noalloc(k, None, gpu.MIXED, -1, d[0].ptr, nt, d[1].ptr, d[2].ptr, d[3].ptr, m,
                                                  o.ptr, 0, ctypes.c_void_p(0)))
        gpu.synchronize()
        # the split partial sums may come in other groups: FP64 rounding of the groups' sums
        assert np.abs(o.download() - out).max() <= 1e-12 * max(np.abs(out).max(), magnitude(k, *a))


@pytest.mark.parametrize("shape", [(100003, 100001), (5003, 2000003), (1500001, 7001)],
                         ids=["square", "few-targets", "few-sources"])
@pytest.mark.parametrize("k", [2, 3, 4])
def test_large_three_outputs(gpu, k, shape):
    """The sizes from which the Stokes layers and the Laplace gradient form their far pairs on the matrix cores:
    against the FP64 Eval (held to the oracle elsewhere), clustered points with coincident ones, with and without
    the FP32 Newton step.  1e-6 normwise, the mixed bar."""
    nt, ns = shape
    rng = np.random.default_rng(nt + k)
    _, K0, K1, _, _ = oracle.dims(k)
    c = rng.random((64, 3))
    xs, xt = (c[rng.integers(0, 64, m)] + 0.05 * rng.standard_normal((m, 3)) for m in (ns, nt))
    xt[:37] = xs[ns - 37:]
    n, v = rng.standard_normal(3 * ns), rng.uniform(-1, 1, K0 * ns)
    d = [gpu.DeviceArray.from_host(a.ravel()) for a in (xt, xs, n, v)]
    res = []
    for prec, flags in ((gpu.FP64, 0), (gpu.MIXED, 0), (gpu.MIXED, gpu.MIXED_NEWTON)):
        o = gpu.DeviceArray.from_host(np.zeros(nt * K1))
        gpu.eval(k, d[0], d[1], d[2], d[3], o, precision=prec, flags=flags)
        gpu.synchronize()
        res.append(o.download())
    for out in res[1:]:
        assert np.isfinite(out).all()
        assert np.abs(out - res[0]).max() <= 1e-6 * np.abs(res[0]).max()
