"""The device eigensolver at the edges of its size classes (one launch up to
64 rows, one workgroup up to 128, meeting workgroups and launched merge
levels up to 512) and on the inputs that take its special branches."""
import numpy as np
import pytest

from itensor_amd.itx import ItxError

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _matrix(kind, n, rng):
    if kind == "random":
        X = rng.standard_normal((n, n))
        return X + X.T
    if kind == "rank":  # density matrix of rank n / 3
        Y = rng.standard_normal((n, max(1, n // 3)))
        return Y @ Y.T / n
    if kind == "decay":  # weights over many decades
        Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        X = (Q * np.exp(-40.0 * np.arange(n) / n)) @ Q.T
        return 0.5 * (X + X.T)
    if kind == "equal":  # two eigenvalues, each many times
        Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        X = (Q * np.where(np.arange(n) % 3 == 0, -2.0, 1.0)) @ Q.T
        return 0.5 * (X + X.T)
    if kind == "diagonal":
        return np.diag(rng.integers(-3, 4, n).astype(float))
    if kind == "blocks":  # zero couplings inside
        X = np.zeros((n, n))
        for a in range(0, n, 7):
            b = min(n, a + 7)
            Y = rng.standard_normal((b - a, b - a))
            X[a:b, a:b] = Y + Y.T
        return X
    if kind == "tiny":
        return 1e-130 * _matrix("random", n, rng)
    return np.zeros((n, n))


def _check(X, w, U):
    n = len(X)
    scale = max(np.abs(np.linalg.eigvalsh(X)).max(), 1e-300)
    tol = 8 * max(n, 8) * EPS  # backward stable: a modest multiple of n eps
    assert np.all(np.diff(w) <= 0)
    assert np.max(np.abs(w - np.linalg.eigvalsh(X)[::-1])) <= tol * scale
    assert np.max(np.abs(U.T @ U - np.eye(n))) <= tol
    assert np.max(np.abs((U * w) @ U.T - X)) <= tol * scale


def _solve(ctx, dev, mats):
    ns = [len(m) for m in mats]
    ao = np.cumsum([0] + [n * n for n in ns])[:-1]
    wo = np.cumsum([0] + ns)[:-1]
    A, w = dev.put(np.concatenate([m.ravel(order="F") for m in mats])), dev.empty(sum(ns))
    wh = ctx.syev_batched_host(ns, ao, A.data_ptr(), wo, w.data_ptr())
    Ah, w = dev.get(A, (A.numel(),)), dev.get(w, (sum(ns),))
    assert np.array_equal(wh[: sum(ns)], w)
    return [(w[o:o + n], Ah[a:a + n * n].reshape((n, n), order="F")) for n, a, o in zip(ns, ao, wo)]


@pytest.mark.parametrize("kind", ["random", "rank", "decay", "equal", "diagonal", "blocks", "tiny", "zero"])
def test_syev_size_classes(ctx, dev, kind):
    rng = np.random.default_rng(len(kind))
    mats = [_matrix(kind, n, rng) for n in (1, 2, 3, 4, 5, 16, 17, 31, 33, 63, 64, 65, 66, 127, 128, 129, 200, 256, 257,
                                            300, 512)]
    for X, (w, U) in zip(mats, _solve(ctx, dev, mats)):
        _check(X, w, U)


def test_syev_more_workgroups_than_cus(ctx, dev):
    """24 matrices of 200 rows: 312 workgroups that meet, two launches."""
    rng = np.random.default_rng(3)
    mats = [_matrix("random", 200, rng) for _ in range(24)] + [_matrix("rank", 30, rng) for _ in range(300)]
    for X, (w, U) in zip(mats, _solve(ctx, dev, mats)):
        _check(X, w, U)


@pytest.mark.parametrize("n", [2, 40, 100, 300])
def test_syev_rejects_not_a_number(ctx, dev, n):
    X = np.eye(n)
    X[n // 2, n // 2] = np.nan
    A, w = dev.put(X), dev.empty(n)
    with pytest.raises(ItxError, match=r"\(5\)"):
        ctx.syev(n, A.data_ptr(), w.data_ptr())
