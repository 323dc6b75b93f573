"""The mixed path's own kernels, above the sizes that run the FP64 ones, for every
micro-kernel at 1, 2 and 4 targets per lane (capped lower by kernels of more
outputs; Laplace FxU and DxU have their one matrix-core form): coincident points
in several tiles, which the unmasked near pairs leave to the tile's second pass,
points far from the origin and scaled, all sources at one point, flat sets.

Tolerance: 1e-6 of the sum of a target's term magnitudes (each FP32 pair is good
to a few 2^-24 of itself), looked at for the eight targets of the largest errors;
the others are bounded by the largest of those sums."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

NT, NS = 1001, 160001


def sets(rng, where):
    xs, xt = rng.random((NS, 3)), rng.random((NT, 3))
    if where == "moved":
        xs, xt = 1e-3 * xs + [2.0, -1.0, 3.0], 1e-3 * xt + [2.0, -1.0, 3.0]
    elif where == "flat":
        xs[:, 1] = xt[:, 1] = -0.5
    elif where == "point":
        xs[:] = xs[0]
        xt[::2] = xs[0]
    xs[5000:5040] = xs[:40]  # sources that coincide with each other too
    xt[3:93] = xs[rng.integers(0, NS, 90)]
    xt[93:103] = xs[5000:5010]
    return xt.ravel(), xs.ravel()


def magnitudes(k, xt, xs, n, v, mu):
    """Sum of |term| per output."""
    K0, out = v.size // NS, 0.0
    for a in range(0, NS, 20000):
        s = slice(3 * a, 3 * (a + 20000))
        out = out + np.abs(oracle.kernel_matrix(k, xt, xs[s], n[s], ctx=mu)).T @ np.abs(v[K0 * a:K0 * (a + 20000)])
    return out


@pytest.mark.parametrize("where", ["cube", "moved", "flat", "point"])
@pytest.mark.parametrize("k", range(16))
def test_own_kernels(gpu, tmp_path, k, where):
    rng = np.random.default_rng(60 + k)
    _, K0, K1, _, _ = oracle.dims(k)
    xt, xs = sets(rng, where)
    n = rng.standard_normal((NS, 3))
    n = (n / np.linalg.norm(n, axis=1)[:, None]).ravel()
    v = rng.uniform(-1, 1, NS * K0)
    mu = 1.0 if k >= 12 else None
    ref = oracle.eval(k, xt, xs, n, v, ctx=mu)
    estimate = gpu.eval(k, xt, xs, n, v, precision=gpu.FP64, digits=7, ctx=mu)  # what the FP64 kernels would give
    gpu.tune_db_path(str(tmp_path / "tpl.db"))
    try:
        for tpl in (1, 2, 4):
            gpu.set_dense_shape(k, NT, NS, tpl, 0, precision=gpu.MIXED)
            out = gpu.eval(k, xt, xs, n, v, precision=gpu.MIXED, ctx=mu)
            assert np.isfinite(out).all()
            err = np.abs(out - ref).reshape(NT, K1)
            worst = np.argsort(err.max(1))[-8:]
            size = magnitudes(k, xt.reshape(-1, 3)[worst].ravel(), xs, n, v, mu).reshape(8, K1).max(1)
            assert (err[worst].max(1) <= 1e-6 * size).all(), tpl
            assert err.max() <= 1e-6 * size.max(), tpl
            assert not np.array_equal(out, estimate)
    finally:
        gpu.tune_db_path(None)
