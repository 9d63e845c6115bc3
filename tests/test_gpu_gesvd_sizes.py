"""The SVD at the edges of its lane groups and of what fits LDS, and at
scales where products of column norms leave the normal range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("m,n,scale", [(2, 300, 1.0), (32, 33, 1.0), (33, 33, 1.0), (64, 64, 1.0), (65, 80, 1.0),
                                       (100, 100, 1.0), (101, 101, 1.0), (129, 131, 1.0), (40, 300, 1.0),
                                       (20, 20, 1e120), (20, 20, 1e-120), (20, 20, 1e-60)])
def test_gesvd_sizes(ctx, dev, m, n, scale):
    rng = np.random.default_rng(m + n)
    M = rng.standard_normal((m, n)) * scale
    M[:, : n // 3] *= 1e-6
    k = min(m, n)
    a, u, s, v = dev.put(M), dev.empty(m * k), dev.empty(k), dev.empty(n * k)
    ctx.gesvd(m, n, a.data_ptr(), u.data_ptr(), s.data_ptr(), v.data_ptr())
    U, S, V = dev.get(u, (m, k)), dev.get(s, (k,)), dev.get(v, (n, k))
    ref = np.linalg.svd(M / scale, compute_uv=False)
    tol = 16 * max(m, n) * EPS  # some ten sweeps of rotations, each a few eps
    assert np.all(np.diff(S) <= 0)
    assert np.max(np.abs(S / scale - ref)) <= tol * ref[0]
    assert np.max(np.abs((U * (S / scale)) @ V.T - M / scale)) <= tol * ref[0]
    assert np.max(np.abs(U.T @ U - np.eye(k))) <= tol
    assert np.max(np.abs(V.T @ V - np.eye(k))) <= tol
