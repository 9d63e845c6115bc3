"""Matrices with exactly dependent columns: what is left of a column shrinks to
denormal squares, and the sweeps end all the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _check(X, U, S, V):
    k = len(S)
    ref = np.linalg.svd(X, compute_uv=False)
    tol = 16 * max(*X.shape, 8) * EPS  # some ten sweeps of rotations, each a few eps
    assert np.all(np.diff(S) <= 0)
    assert np.max(np.abs(S - ref)) <= tol * ref[0]
    assert np.max(np.abs((U * S) @ V.T - X)) <= tol * ref[0]
    big = S > 1e-12 * ref[0]  # the long side's columns of the others are noise or zero
    long, short = (U, V) if X.shape[0] > X.shape[1] else (V, U)  # a square matrix counts as wide
    assert np.max(np.abs(short.T @ short - np.eye(k))) <= tol
    assert np.max(np.abs((long.T @ long)[np.ix_(big, big)] - np.eye(big.sum()))) <= tol


@pytest.mark.parametrize("scale", [1.0, 1e100, 1e-100])
@pytest.mark.parametrize("kind", ["rank-one", "sparse", "repeated"])
def test_gesvd_dependent_columns(ctx, dev, kind, scale):
    rng = np.random.default_rng(len(kind))
    M = []
    for i in range(250):  # below the count from which small matrices are treated apart
        m, n = rng.integers(2, 50, 2)
        if kind == "rank-one":
            X = np.linalg.qr(rng.standard_normal((m, m)))[0] @ np.ones((m, n))
        elif kind == "sparse":
            X = rng.standard_normal((m, n)) * (rng.random((m, n)) < 0.1)
            X[0, 0] = 1.0
        else:
            X = rng.standard_normal((m, n))[:, rng.integers(0, max(1, n // 3), n)]
        M.append(X)
    m, n = np.array([x.shape for x in M]).T
    k = np.minimum(m, n)
    ao, uo, so, vo = (np.concatenate([[0], np.cumsum(x)])[:-1] for x in (m * n, m * k, k, n * k))
    a = dev.put(np.concatenate([(scale * x).ravel(order="F") for x in M]))
    u, s, v = dev.empty((m * k).sum()), dev.empty(k.sum()), dev.empty((n * k).sum())
    ctx.gesvd_batched(m, n, ao, a.data_ptr(), uo, u.data_ptr(), so, s.data_ptr(), vo, v.data_ptr())
    u, s, v = (dev.get(t, (t.numel(),)) for t in (u, s, v))
    for i, X in enumerate(M):
        U = u[uo[i]:uo[i] + m[i] * k[i]].reshape((m[i], k[i]), order="F")
        V = v[vo[i]:vo[i] + n[i] * k[i]].reshape((n[i], k[i]), order="F")
        _check(X, U, s[so[i]:so[i] + k[i]] / scale, V)
