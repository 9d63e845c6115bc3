"""The workgroups that reduce one matrix together wait for each other within a
bound; a matrix whose workgroups did not meet takes the path without meetings.
ITX_EIG_WAIT shortens the bound, or leaves a workgroup out, from the host."""
import time

import numpy as np
import pytest

from test_gpu_syev_dc import _check, _matrix, _solve

pytestmark = pytest.mark.gpu


def test_missing_workgroup_costs_one_bound(ctx, dev, monkeypatch):
    """300 rows: 19 workgroups, one of them never launched, whose columns every
    one of the 298 steps waits for.  A bound of 2^15 polls is some 30 ms and the
    path without meetings another 30; a bound per step would be seconds."""
    rng = np.random.default_rng(5)
    mats = [_matrix("random", n, rng) for n in (300, 40, 130, 100)]
    _solve(ctx, dev, mats)
    monkeypatch.setenv("ITX_EIG_WAIT", f"{1 << 15},1")
    t = time.perf_counter()
    got = _solve(ctx, dev, mats)
    t = time.perf_counter() - t
    for X, (w, U) in zip(mats, got):
        _check(X, w, U)
    assert t < 0.5
