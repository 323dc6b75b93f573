"""Near lists at the sizes where a build takes other paths, against the oracle's
brute force (integers and copied coordinates, equal): more near elements per
target than its buffers are first sized for (8 and 24), pair keys of more than
32 bits, elements of more than 4096 nodes (several 64-node chunks per node box),
and numbers of pairs around powers of two, where the sorts change algorithm."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def same(got, want):
    assert want["near_scatter_index"].size > 0
    for k, w in want.items():
        assert (w is None and got[k] is None) or np.array_equal(got[k], w), k


def check(gpu, xt, xs, rad, cnt, normals=False):
    dsp = np.concatenate(([0], np.cumsum(cnt)[:-1]))
    xn = np.random.default_rng(7).standard_normal(xt.size) if normals else None
    got = gpu.near_list(xt, xs, rad, cnt, dsp, Xn_trg=xn)
    want = oracle.default().near_list(xt, xs, rad, cnt, dsp, Xn_trg=xn)
    same(got, want)
    return want["near_scatter_index"].size


@pytest.mark.parametrize("nt,nelem", [(9000, 12), (3001, 40), (2000, 64)])
def test_many_near_elements_per_target(gpu, nt, nelem):
    """Every target near (almost) every element: 12 to 64 pairs per target."""
    rng = np.random.default_rng(nt)
    cnt = rng.integers(1, 9, nelem)
    n = check(gpu, rng.random(3 * nt), rng.random(3 * cnt.sum()), rng.uniform(1.2, 2.0, cnt.sum()), cnt, normals=True)
    assert n > 10 * nt


def test_wide_keys(gpu):
    """70 001 targets (17 bits) and 40 003 elements (16 bits) of one node."""
    rng = np.random.default_rng(2)
    cnt = np.ones(40003, dtype=np.int64)
    check(gpu, rng.random(3 * 70001), rng.random(3 * 40003), rng.uniform(0.0, 0.02, 40003), cnt)


def test_large_elements(gpu):
    """Node boxes of 64, 128 and 192 nodes, radii that reach a few nodes or thousands."""
    rng = np.random.default_rng(3)
    cnt = np.array([4096, 4097, 70, 10007, 1, 8192])
    c = np.repeat(rng.random((cnt.size, 3)), cnt, axis=0)
    xs = (c + 0.1 * rng.standard_normal(c.shape)).ravel()
    check(gpu, rng.random(3 * 6000), xs, 10.0 ** rng.uniform(-3, -0.7, cnt.sum()), cnt)


@pytest.mark.parametrize("n", [1, 63, 1024, 4095, 65536, 65537, 70000])
def test_numbers_of_pairs(gpu, n):
    """n targets at one element's node, as many far away."""
    rng = np.random.default_rng(n)
    xt = np.concatenate([0.5 + 1e-3 * rng.uniform(-1, 1, (n, 3)), 0.4 * rng.random((n, 3))])
    xt = xt[rng.permutation(2 * n)].ravel()
    assert check(gpu, xt, np.array([0.5, 0.5, 0.5]), np.array([0.01]), np.array([1])) == n
