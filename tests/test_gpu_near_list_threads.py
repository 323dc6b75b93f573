"""Near lists built by several threads at once (each on its own per-thread
stream), over and over with buffers of different sizes that are kept between
builds, give the lists that one thread gives; so do lists that are read after
others were built and destroyed."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(seed, nelem, nt):
    rng = np.random.default_rng(seed)
    cnt = rng.integers(1, 130, nelem)
    dsp = np.concatenate(([0], np.cumsum(cnt)[:-1]))
    centre = rng.random((nelem, 3))
    xs = np.repeat(centre, cnt, axis=0) + 0.02 * rng.standard_normal((cnt.sum(), 3))
    return rng.random(3 * nt), xs.ravel(), rng.uniform(0.01, 0.08, cnt.sum()), cnt, dsp


def test_threads(gpu):
    cases = [case(i, 20 + 130 * (i % 3), 500 * (1 + 7 * (i % 4))) for i in range(12)]
    want = [gpu.near_list(*c) for c in cases]

    def build(i):
        return i, gpu.near_list(*cases[i])

    with ThreadPoolExecutor(4) as pool:
        for i, got in pool.map(build, list(range(12)) * 5):
            for key, value in want[i].items():
                assert (value is None and got[key] is None) or np.array_equal(got[key], value), (i, key)
