"""FP64 Evals at full precision keep the KernelMatrix's accuracy where few sources
leave nothing to average: one source of density 1, whose Eval takes the same
operations as its matrix entry, so its rms error against long double is the
entry's (within 5 %; the rsqrt that rounds twice at full size gives 18 % more,
rounding f n in place of n.r 29 %).  And both sides of the number of sources from
which the shorter forms are used, against the oracle: 2e-14 of the largest sum of
magnitudes (600 terms of 2^-53 each, relative to their sizes, at most 6e-14 / 3)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
L = np.longdouble
PI = L("3.14159265358979323846264338327950288")


@pytest.mark.parametrize("how", ["eval", "dense_plan", "plan"])
@pytest.mark.parametrize("k", [0, 1, 4])
def test_one_source(gpu, k, how):
    if k == 1 and how == "plan":
        pytest.skip("batched plans stage f n for every block")
    rng = np.random.default_rng(k)
    nt = 20000
    xt, xs, n, f = rng.random((nt, 3)), rng.random((1, 3)), rng.standard_normal((1, 3)), np.ones(1)
    d = xt.astype(L) - xs.astype(L)
    z = 1 / np.sqrt((d * d).sum(-1))
    want = {0: lambda: z[:, None], 1: lambda: ((d * n).sum(-1) * z ** 3)[:, None], 4: lambda: -d * (z ** 3)[:, None]}[k]()
    want = want / (4 * PI)
    K1 = want.shape[1]
    a = (xt.ravel(), xs.ravel(), n.ravel())
    M = gpu.kernel_matrix(k, *a).reshape(nt, K1)
    if how == "eval":
        out = gpu.eval(k, *a, f)
    elif how == "dense_plan":
        out = gpu.DensePlan(k, *a).apply(f)
    else:
        P = gpu.Plan(k, [0], [nt], [0], [1], nt, 1)
        P.set_geometry(*a)
        out = P.apply(f, np.zeros(nt * K1))
    rms = [float(np.sqrt((((q.reshape(nt, K1).astype(L) - want) / np.abs(want)) ** 2).mean())) for q in (out, M)]
    assert rms[0] <= 1.05 * rms[1], rms


@pytest.mark.parametrize("ns", [1, 255, 511, 512, 513, 600])
@pytest.mark.parametrize("k", [0, 1, 3, 4, 7, 10])
def test_both_forms(gpu, k, ns):
    rng = np.random.default_rng(ns)
    _, K0, K1, _, _ = oracle.dims(k)
    nt = 1033
    xt, xs, n, v = rng.random(3 * nt), rng.random(3 * ns), rng.standard_normal(3 * ns), rng.standard_normal(K0 * ns)
    xt[:3] = xs[-3:]
    ref = oracle.eval(k, xt, xs, n, v)
    size = np.max(np.abs(oracle.kernel_matrix(k, xt, xs, n)).T @ np.abs(v))
    out = gpu.eval(k, xt, xs, n, v)
    assert np.abs(out - ref).max() <= 2e-14 * size
    assert np.array_equal(gpu.DensePlan(k, xt, xs, n).apply(v), out)


@pytest.mark.parametrize("k", [0, 1, 3, 4, 7, 10])
def test_blocks_of_both_forms(gpu, k):
    """A plan whose blocks' lanes sum fewer and more sources than that, in one piece and in several, with one, two and
    four lane groups."""
    rng = np.random.default_rng(k)
    _, K0, K1, _, _ = oracle.dims(k)
    tc = np.array([128, 128, 5, 20, 30, 16, 128, 50, 300])
    sc = np.array([511, 512, 513, 2047, 2048, 2049, 5000, 1024, 1])
    td, sd = (np.concatenate(([0], np.cumsum(a)[:-1])) for a in (tc, sc))
    xt, xs, n = rng.random(3 * tc.sum()), rng.random(3 * sc.sum()), rng.standard_normal(3 * sc.sum())
    v = rng.standard_normal(K0 * sc.sum())
    for b in range(tc.size):  # a coincident pair in each block
        xt[3 * td[b]:3 * td[b] + 3] = xs[3 * (sd[b] + sc[b]) - 3:3 * (sd[b] + sc[b])]
    P = gpu.Plan(k, td, tc, sd, sc, int(tc.sum()), int(sc.sum()))
    P.set_geometry(xt, xs, n)
    for tpl in (2, 1):
        P.set_shape(2, tpl, 0)
        out = P.apply(v, np.zeros(K1 * tc.sum()))
        for b in range(tc.size):
            t, s = slice(3 * td[b], 3 * (td[b] + tc[b])), slice(3 * sd[b], 3 * (sd[b] + sc[b]))
            f = v[K0 * sd[b]:K0 * (sd[b] + sc[b])]
            ref = oracle.eval(k, xt[t], xs[s], n[s], f)
            size = np.max(np.abs(oracle.kernel_matrix(k, xt[t], xs[s], n[s])).T @ np.abs(f))
            # 5000 terms in sums of at most 128, their roundings relative to partial sums
            assert np.abs(out[K1 * td[b]:K1 * (td[b] + tc[b])] - ref).max() <= 2e-14 * size, (tpl, b)
