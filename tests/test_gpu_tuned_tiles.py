"""Entries of the tile table that a contraction of the same size class cannot
use: the contraction is planned as if there were none."""
import numpy as np
import pytest

from itensor_amd.itx import Context

pytestmark = pytest.mark.gpu
EPS = {"f64": np.finfo(float).eps, "f32": np.finfo(np.float32).eps, "bf16x3": 2.0**-14}


@pytest.fixture
def own(torch_dev):
    import torch

    c = Context(0, torch.cuda.current_stream().cuda_stream)
    yield c
    c.close()


def _table(ctx, tmp_path, tile, prec, M, N, K, akc=1, bkc=1):
    lg = [int(np.ceil(np.log2(x))) for x in (M, N, K)]
    p = {"f64": 0, "f32": 1, "bf16x3": 2}[prec]
    path = tmp_path / "tiles"
    path.write_text("p%d a%d b%d M%d N%d K%d G0|%d\n" % (p, akc, bkc, *lg, tile))
    ctx.tune_load(str(path))


def _contract(ctx, dev, M, N, K, prec):
    rng = np.random.default_rng(M + N + K)
    A, B = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    a, b, c = dev.put(A.T), dev.put(B), dev.empty(M * N)
    p = ctx.plan_dense((K, M), (-1, 1), (K, N), (-1, 2), (M, N), (1, 2), prec)
    p.execute(a.data_ptr(), b.data_ptr(), c.data_ptr())
    bound = (K + 70) * EPS[prec] * (np.abs(A) @ np.abs(B))
    assert np.all(np.abs(dev.get(c, (M, N)) - A @ B) <= bound)
    return p.info["tile"]


@pytest.mark.parametrize("prec,tile", [("f64", 14), ("f64", 15), ("f32", 14), ("f32", 15), ("f64", 18), ("bf16x3", 14),
                                       ("bf16x3", 18), ("f64", 5), ("f64", 99), ("f64", -1)])
def test_table_entry_of_another_alignment(own, dev, tmp_path, prec, tile):
    M, N, K = 255, 253, 129  # odd: operands in single loads
    untuned = _contract(own, dev, M, N, K, prec)
    _table(own, tmp_path, tile, prec, M, N, K)
    assert _contract(own, dev, M, N, K, prec) == untuned


@pytest.mark.parametrize("prec,tile", [("f64", 14), ("f64", 17), ("f32", 14), ("f32", 16), ("bf16x3", 4), ("f64", 10)])
def test_table_entry_that_fits(own, dev, tmp_path, prec, tile):
    _table(own, tmp_path, tile, prec, 256, 252, 132)
    assert _contract(own, dev, 256, 252, 132, prec) == tile


def test_tuned_class_serves_odd_sizes(own, dev):
    """The tuner measures an aligned size; an odd one of its class follows."""
    own.set_autotune(True)
    assert _contract(own, dev, 256, 252, 132, "f64") not in (14, 15)
    n = own.tune_size()
    _contract(own, dev, 255, 253, 129, "f64")
    assert own.tune_size() == n
