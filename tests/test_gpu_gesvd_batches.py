"""More small matrices than CUs take a kernel of four waves each: at the edges
of its lane groups, beside larger matrices in the same call, and either side
of the count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
SIZES = [(1, 1), (3, 64), (8, 8), (9, 7), (9, 9), (16, 17), (17, 17), (32, 64), (33, 33), (64, 63), (64, 64), (0, 5), (5, 12)]


def _batch(ctx, dev, shapes):
    rng = np.random.default_rng(len(shapes))
    M = [rng.standard_normal(s) for s in shapes]
    for x in M:
        x[:, : x.shape[1] // 3] *= 1e-6
    m, n = np.array(shapes).T
    k = np.minimum(m, n)
    ao, uo, so, vo = (np.concatenate([[0], np.cumsum(x)])[:-1] for x in (m * n, m * k, k, n * k))
    a = dev.put(np.concatenate([x.ravel(order="F") for x in M]))
    u, s, v = dev.empty((m * k).sum()), dev.empty(k.sum()), dev.empty((n * k).sum())
    ctx.gesvd_batched(m, n, ao, a.data_ptr(), uo, u.data_ptr(), so, s.data_ptr(), vo, v.data_ptr())
    u, s, v = (dev.get(t, (t.numel(),)) for t in (u, s, v))
    for i, x in enumerate(M):
        if k[i] == 0:
            continue
        U = u[uo[i]:uo[i] + m[i] * k[i]].reshape((m[i], k[i]), order="F")
        V = v[vo[i]:vo[i] + n[i] * k[i]].reshape((n[i], k[i]), order="F")
        S = s[so[i]:so[i] + k[i]]
        ref = np.linalg.svd(x, compute_uv=False)
        tol = 16 * max(m[i], n[i], 8) * EPS  # some ten sweeps of rotations, each a few eps
        assert np.all(np.diff(S) <= 0)
        assert np.max(np.abs(S - ref)) <= tol * ref[0]
        assert np.max(np.abs((U * S) @ V.T - x)) <= tol * ref[0]
        assert np.max(np.abs(U.T @ U - np.eye(k[i]))) <= tol
        assert np.max(np.abs(V.T @ V - np.eye(k[i]))) <= tol


@pytest.mark.parametrize("extra", [[], [(65, 20), (100, 100), (20, 300), (102, 101)]], ids=["small", "mixed"])
def test_gesvd_many_small(ctx, dev, extra):
    _batch(ctx, dev, (SIZES * 30 + extra * 2)[::-1])


@pytest.mark.parametrize("over", [0, 1])
def test_gesvd_count(ctx, dev, over):
    _batch(ctx, dev, [(12, 9)] * (ctx.cus + over))
