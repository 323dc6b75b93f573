"""Host Evals whose arrays just fit, and just do not fit, one pinned staging
chunk (8 MiB): the same bits as the Eval on device arrays, accumulated into
v_trg, FP64 and mixed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,words", [(0, 4), (3, 9)])
@pytest.mark.parametrize("over", [-64, 0, 64])
def test_chunk_edge(gpu, k, words, over):
    nt = 70
    _, K0, K1, ND, _, _, _ = gpu.kernel_info(k)
    ns = ((8 << 20) // 8 - nt * (3 + K1) - 5 * 32) // words + over
    rng = np.random.default_rng(ns)
    xt, xs, n, v = rng.random(3 * nt), rng.random(3 * ns), rng.standard_normal(3 * ns), rng.uniform(-1, 1, K0 * ns)
    start = rng.standard_normal(nt * K1)
    for prec in (gpu.FP64, gpu.MIXED):
        d = [gpu.DeviceArray.from_host(a) for a in (xt, xs, n, v, start)]
        gpu.eval(k, *d, precision=prec)
        gpu.synchronize()
        out = gpu.eval(k, xt, xs, n, v, start.copy(), precision=prec)
        assert np.array_equal(out, d[4].download())
