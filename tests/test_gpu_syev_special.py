"""The device eigensolver on entries outside the range of ordinary arithmetic,
in one call with ordinary matrices."""
import numpy as np
import pytest

from itensor_amd.itx import ItxError
from test_gpu_syev_dc import _check, _matrix, _solve

pytestmark = pytest.mark.gpu


def _check_diagonal(d, w, U):
    """Exactly d in descending order, and the unit vectors that go with it."""
    order = np.argsort(-d, kind="stable")
    assert np.array_equal(w, d[order], equal_nan=True)
    at = np.argmax(np.abs(U), axis=0)
    assert np.array_equal(np.sort(at), np.arange(len(d)))
    assert np.array_equal(np.abs(U), np.eye(len(d))[:, at])
    assert np.array_equal(d[at], w, equal_nan=True)


@pytest.mark.parametrize("x", [np.nan, np.inf, -np.inf, -3.0, 0.0, 5e-324])
def test_syev_single_row(ctx, dev, x):
    rng = np.random.default_rng(1)
    mats = [np.array([[x]]), _matrix("random", 40, rng), np.array([[x]]), _matrix("random", 130, rng)]
    got = _solve(ctx, dev, mats) if x == x else None
    if got is None:  # the comparison of w and its host copy fails on not-a-number
        A, w = dev.put(np.array([[x]])), dev.empty(1, fill=0.0)
        ctx.syev(1, A.data_ptr(), w.data_ptr())
        assert np.isnan(dev.get(w, (1,))[0]) and abs(dev.get(A, (1,))[0]) == 1.0
        return
    for X, (w, U) in zip(mats, got):
        if len(X) == 1:
            _check_diagonal(np.diag(X), w, U)
        else:
            _check(X, w, U)


@pytest.mark.parametrize("n", [2, 3, 40, 64, 65, 100, 129, 200, 300])
def test_syev_infinite_diagonal(ctx, dev, n):
    rng = np.random.default_rng(n)
    d = rng.permutation(np.arange(n) - n / 3.0)
    d[rng.integers(n)] = np.inf
    e = d.copy()
    e[rng.integers(n)] = -np.inf
    X = _matrix("random", 50, rng)
    for M, (w, U) in zip((d, X, e), _solve(ctx, dev, [np.diag(d), X, np.diag(e)])):
        if M is X:
            _check(X, w, U)
        else:
            _check_diagonal(M, w, U)


@pytest.mark.parametrize("n", [1, 2, 40, 100, 200])
def test_syev_largest_numbers(ctx, dev, n):
    """Entries of 2^1023 and more, whose scale as a power of two would not be a number."""
    d = np.linspace(-1.75, 1.75, n) if n > 1 else np.array([1.5])
    (w, U), = _solve(ctx, dev, [np.diag(d) * 2.0**1023])
    assert np.array_equal(w, np.sort(d)[::-1] * 2.0**1023)
    if n > 1:
        (w, U), = _solve(ctx, dev, [np.array([[1.0, 0.25], [0.25, 1.0]]) * 2.0**1023])
        assert np.max(np.abs(w * 2.0**-1023 - [1.25, 0.75])) <= 64 * np.finfo(float).eps


def _rank_one(n):
    return np.ones((n, n))


def _graded(n):
    rng = np.random.default_rng(n)
    d = 10.0 ** (-0.4 * np.arange(n))
    Y = rng.standard_normal((n, n))
    return d[:, None] * (Y + Y.T) * d


def _graded_up(n):
    return _graded(n)[::-1, ::-1].copy()


@pytest.mark.parametrize("wait", [None, "0"])
@pytest.mark.parametrize("scale", [1.0, 1e-140, 1e140, 1e-250, 1e250])
@pytest.mark.parametrize("make", [_rank_one, _graded, _graded_up, lambda n: _matrix("random", n, np.random.default_rng(n)),
                                  lambda n: np.eye(n) + 1e-15 * _matrix("random", n, np.random.default_rng(n))],
                         ids=["rank-one", "graded", "graded-up", "random", "identity"])
def test_syev_squares_out_of_range(ctx, dev, monkeypatch, make, scale, wait):
    """Columns whose squares are no numbers: what is left of a column when the
    rank or the grading has used it up, and whole matrices of such a scale."""
    if wait is not None:
        monkeypatch.setenv("ITX_EIG_WAIT", wait)
    mats = [make(n) * scale for n in (2, 3, 24, 64, 65, 128, 153, 200, 256, 300, 400)]
    for X, (w, U) in zip(mats, _solve(ctx, dev, mats)):
        _check(X / scale, w / scale, U)


@pytest.mark.parametrize("n", [100, 129, 200, 300])
def test_syev_infinite_coupling(ctx, dev, n):
    """No decomposition: an error or the diagonal, and the context keeps working.
    (An infinite coupling of a merge once gave an eigenvalue that is not a
    number, whose place in the order was never written.)"""
    d, e = np.linspace(1.0, 2.0, n), np.zeros(n - 1)
    e[n // 2 - 1] = np.inf
    X = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    try:
        (w, U), = _solve(ctx, dev, [X])
        assert np.array_equal(w, d[::-1])
    except ItxError as err:
        assert "(5)" in str(err)
    rng = np.random.default_rng(n)
    Y = _matrix("random", n, rng)
    (w, U), = _solve(ctx, dev, [Y])
    _check(Y, w, U)
