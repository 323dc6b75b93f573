"""The matrix-core form of the Stokes double layer and the Laplace gradient is no
less exact than the FP32 form, for sets apart (all pairs far): the whole Eval,
which takes the matrix cores, against the same sum in pieces of sources small
enough for the FP32 form, errors against the FP64 Eval, geometric mean over eight
draws.  5 % more is allowed for the pieces' other tiles and the draws."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [3, 4])
def test_sets_apart(gpu, k):
    nt, ns, piece = 100003, 100001, 9001
    _, K0, K1, _, _, _, _ = gpu.kernel_info(k)
    err = np.zeros((8, 2))
    for seed in range(8):
        rng = np.random.default_rng(seed)
        xt, xs = 3.0 + 0.2 * rng.random(3 * nt), rng.random(3 * ns)
        n = rng.standard_normal((ns, 3))
        n, v = (n / np.linalg.norm(n, axis=1)[:, None]).ravel(), rng.uniform(-1, 1, K0 * ns)
        t = gpu.DeviceArray.from_host(xt)
        res = []
        for prec, step in ((gpu.FP64, ns), (gpu.MIXED, ns), (gpu.MIXED, piece)):
            out = gpu.DeviceArray.from_host(np.zeros(nt * K1))
            for a in range(0, ns, step):
                s = slice(3 * a, 3 * (a + step))
                d = [gpu.DeviceArray.from_host(q) for q in (xs[s], n[s], v[K0 * a:K0 * (a + step)])]
                gpu.eval(k, t, d[0], d[1], d[2], out, precision=prec)
                gpu.synchronize()
            res.append(out.download())
        err[seed] = [np.linalg.norm(q - res[0]) / np.linalg.norm(res[0]) for q in res[1:]]
    whole, pieces = np.exp(np.log(err).mean(0))
    print("matrix cores %.3e, FP32 form in pieces %.3e" % (whole, pieces))
    assert whole <= 1.05 * pieces
