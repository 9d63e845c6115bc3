"""The workgroups that reduce one matrix together wait for each other within a
bound; a matrix whose workgroups did not meet takes the path without meetings.
ITX_EIG_WAIT shortens the bound, or leaves a workgroup out, from the host."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from conftest import ROOT
from itensor_amd.itx import ItxError
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


@pytest.mark.parametrize("kind", ["random", "rank", "decay", "equal", "diagonal", "blocks", "zero"])
def test_matrices_that_did_not_meet(ctx, dev, monkeypatch, kind):
    """Every wait given up at once: the matrices above 128 rows start again from
    A on the other path, beside those whose results stand."""
    rng = np.random.default_rng(len(kind))
    mats = [_matrix(kind, n, rng) for n in (200, 30, 129, 1, 128, 512, 64, 300, 257)]
    monkeypatch.setenv("ITX_EIG_WAIT", "0")
    for X, (w, U) in zip(mats, _solve(ctx, dev, mats)):
        _check(X, w, U)


def test_did_not_meet_not_a_number(ctx, dev, monkeypatch):
    monkeypatch.setenv("ITX_EIG_WAIT", "0")
    X = np.eye(200)
    X[100, 100] = np.nan
    A, w = dev.put(X), dev.empty(200)
    with pytest.raises(ItxError, match=r"\(5\)"):
        ctx.syev(200, A.data_ptr(), w.data_ptr())


OWN = """
import numpy as np, torch
import itensor_amd
from itensor_amd.itx import Context
from conftest import Dev
from test_gpu_syev_dc import _check, _matrix, _solve
ctx = Context(0, torch.cuda.current_stream().cuda_stream)
rng = np.random.default_rng(9)
mats = [_matrix(k, n, rng) for k, n in (("random", 600), ("rank", 40), ("blocks", 513), ("decay", 150))]
for X, (w, U) in zip(mats, _solve(ctx, Dev(torch.device("cuda:0")), mats)):
    _check(X, w, U)
print("solved", flush=True)
"""


@pytest.mark.parametrize("wait", [None, "0"])
def test_own_kernels_above_512_rows(torch_dev, wait):
    """ITX_EIG_OWN is read once, so a process of its own: the cooperative
    reduction (and with `wait` the single workgroups beside it)."""
    env = dict(os.environ, ITX_EIG_OWN="1", PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    if wait is not None:
        env["ITX_EIG_WAIT"] = wait
    r = subprocess.run([sys.executable, "-c", OWN], env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "solved" in r.stdout, r.stderr[-2000:]
