"""Near-field matrices and their GEMV where a block's columns are cut into
pieces: one to a few blocks with many sources, odd counts around the 64-column
chunks and the shortest pieces, matrix rows that start at any offset within a
line, nothing written outside the blocks' rows, store and subtract, and with
the target normal; against weighted kernel matrices of the oracle.

Tolerance: 1e-13 normwise (1e-13 of the sum of magnitudes for the GEMV)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 63, 128, 129, 191, 700, 2049])
@pytest.mark.parametrize("k,ndot", [(0, False), (1, False), (3, False), (3, True), (6, False), (4, True)])
def test_pieces(gpu, k, ndot, ns):
    rng = np.random.default_rng(ns + 31 * k)
    _, K0, K1, _, _ = oracle.dims(k)
    dof = K1 // 3 if ndot else K1
    tc, sc = np.array([19, 3, 33]), np.array([ns, 5, ns + 66])
    td, sd = np.concatenate(([0], np.cumsum(tc)[:-1])), np.concatenate(([0], np.cumsum(sc)[:-1]))
    xt, xs = rng.random(3 * tc.sum()), rng.random(3 * sc.sum())
    xt[:3] = xs[3 * (ns - 1):3 * ns]
    xn, tn = rng.standard_normal(xs.size), rng.standard_normal(xt.size)
    w = rng.random(sc.sum())
    size = tc * dof * sc * K0
    off = np.array([5, -1, 5 + size[0] + 7])  # the second block has no matrix
    plan = gpu.Plan(k, td, tc, sd, sc, int(tc.sum()), int(sc.sum()))
    plan.set_geometry(xt, xs, xn)
    length = plan.near_layout(off, trg_normal_dot=ndot)
    before = rng.standard_normal(length + 16)
    want, mat = before.copy(), {}
    for b in (0, 2):
        t, s = slice(3 * td[b], 3 * (td[b] + tc[b])), slice(3 * sd[b], 3 * (sd[b] + sc[b]))
        M = oracle.kernel_matrix(k, xt[t], xs[s], xn[s]).reshape(sc[b] * K0, tc[b], K1)
        if ndot:
            M = (M.reshape(sc[b] * K0, tc[b], dof, 3) * tn[t].reshape(1, tc[b], 1, 3)).sum(-1)
        M = M.reshape(sc[b] * K0, tc[b] * dof).T * np.repeat(w[sd[b]:sd[b] + sc[b]], K0)[None]
        mat[b] = M
        want[off[b]:off[b] + size[b]] -= M.ravel()
    K = before.copy()
    plan.near_matrix(K, w, tn if ndot else None, gpu.NEAR_SUBTRACT)
    scale = max(np.abs(want).max(), max(np.abs(m).max() for m in mat.values()))
    assert np.abs(K - want).max() <= 1e-13 * scale
    outside = np.ones(K.size, bool)
    for b in (0, 2):
        outside[off[b]:off[b] + size[b]] = False
    assert np.array_equal(K[outside], before[outside])
    plan.near_matrix(K, w, tn if ndot else None, gpu.NEAR_STORE)
    for b in (0, 2):
        assert np.abs(K[off[b]:off[b] + size[b]] - mat[b].ravel()).max() <= 1e-13 * np.abs(mat[b]).max()
    F = rng.standard_normal(K0 * sc.sum())
    U = plan.near_gemv(K, F, np.full(tc.sum() * dof, 7.0))
    for b in range(3):
        u = U[td[b] * dof:(td[b] + tc[b]) * dof]
        if b == 1:
            assert (u == 0).all()
            continue
        f = F[sd[b] * K0:(sd[b] + sc[b]) * K0]
        assert np.abs(u - mat[b] @ f).max() <= 1e-13 * (np.abs(mat[b]) @ np.abs(f)).max()
