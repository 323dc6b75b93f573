"""Plans whose blocks have long source ranges: a chunk of targets is cut into
pieces of the sources and the pieces' sums are added up.  Few targets (lane
groups) and a ragged last chunk, one piece to forty, applied twice into the
same output, against the oracle.

Tolerances, normwise: FP64 1e-13; mixed 1e-6 (the bars of the other tests).
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [64, 127, 129, 1000, 5001])
@pytest.mark.parametrize("nt", [1, 17, 40, 129])
@pytest.mark.parametrize("k", [1, 3])
def test_pieces(gpu, k, nt, ns):
    rng = np.random.default_rng(7 * nt + ns + k)
    _, K0, K1, _, _ = oracle.dims(k)
    sizes_t, sizes_s = np.array([nt, 5, nt + 3]), np.array([ns, 70, 33])
    td, sd = np.concatenate(([0], np.cumsum(sizes_t)[:-1])), np.concatenate(([0], np.cumsum(sizes_s)[:-1]))
    xt, xs = rng.random(3 * sizes_t.sum()), rng.random(3 * sizes_s.sum())
    xt[:3] = xs[3 * (ns - 1):3 * ns]  # coincident with the first block's last source
    n = rng.standard_normal(xs.size)
    v = rng.uniform(-1, 1, K0 * sizes_s.sum())
    ref = np.concatenate([oracle.eval(k, xt[3 * a:3 * (a + ta)], xs[3 * b:3 * (b + sb)], n[3 * b:3 * (b + sb)],
                                      v[K0 * b:K0 * (b + sb)]) for a, ta, b, sb in zip(td, sizes_t, sd, sizes_s)])
    for prec, tol in ((gpu.FP64, 1e-13), (gpu.MIXED, 1e-6)):
        plan = gpu.Plan(k, td, sizes_t, sd, sizes_s, int(sizes_t.sum()), int(sizes_s.sum()), precision=prec)
        plan.set_geometry(xt, xs, n)
        out = np.zeros(K1 * sizes_t.sum())
        plan.apply(v, out)
        plan.apply(v, out)
        assert np.abs(out - 2 * ref).max() <= 2 * tol * np.abs(ref).max(), prec
