"""FP64 Eval where its source range is cut into pieces shorter than a staged
tile: odd numbers of sources around the piece (64) and the tile (256), with
coincident points, through sctl_amd_eval and a dense plan, against the oracle.

Tolerance: 1e-13 normwise, the FP64 bar of the other tests (every pair is good
to a few 2^-53 and at most 770 of them are summed).
"""
import numpy as np
import pytest

import oracle
from sctl_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 2, 63, 64, 65, 127, 255, 256, 257, 321, 769])
@pytest.mark.parametrize("nt", [1, 255, 513])
def test_short_splits(gpu, nt, ns):
    rng = np.random.default_rng(1000 * nt + ns)
    for k in (0, 1, 3, 6):
        _, K0, K1, _, _ = oracle.dims(k)
        xs, xt = rng.random(3 * ns), rng.random(3 * nt)
        m = 3 * min(nt, ns, 5)
        xt[:m] = xs[3 * ns - m:]  # coincident with the last sources
        n = rng.standard_normal(3 * ns)
        v = rng.uniform(-1, 1, K0 * ns)
        ref = oracle.eval(k, xt, xs, n, v)
        tol = 1e-13 * max(np.abs(ref).max(), 1e-300)
        out = gpu.eval(k, xt, xs, n, v)
        assert np.abs(out - ref).max() <= tol, (k, W.rel_errors(out, ref))
        plan = gpu.DensePlan(k, xt, xs, n)
        assert np.array_equal(plan.apply(v), out), k


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 129, 769])
def test_short_splits_helmholtz(gpu, ns):
    """The Helmholtz kernels, whose tiles are as long as the shortest piece; same tolerance."""
    nt, mu = 257, 3.0
    rng = np.random.default_rng(ns)
    for k in (12, 13, 14, 15):
        _, K0, K1, _, _ = oracle.dims(k)
        xs, xt = rng.random(3 * ns), rng.random(3 * nt)
        m = 3 * min(nt, ns, 5)
        xt[:m] = xs[3 * ns - m:]
        n = rng.standard_normal(3 * ns)
        v = rng.uniform(-1, 1, K0 * ns)
        ref = oracle.eval(k, xt, xs, n, v, ctx=mu)
        tol = 1e-13 * max(np.abs(ref).max(), 1e-300)
        out = gpu.eval(k, xt, xs, n, v, ctx=mu)
        assert np.abs(out - ref).max() <= tol, (k, W.rel_errors(out, ref))
        plan = gpu.DensePlan(k, xt, xs, n, ctx=mu)
        assert np.array_equal(plan.apply(v), out), k
