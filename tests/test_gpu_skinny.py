"""The skinny contraction path at the edges of its variants: 16-column
groups, k chunks of 20, 256-row units, more units than resident workgroups
and several tasks per C block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("M,N,K,beta", [(256, 1, 1, 0.0), (257, 16, 20, 0.5), (511, 17, 21, 0.0), (1000, 32, 64, -1.0),
                                        (300, 20, 19, 0.0), (200100, 32, 20, 0.0), (200100, 5, 40, 0.25)])
@pytest.mark.parametrize("order", ["km", "mk"])
def test_skinny_dense(ctx, dev, M, N, K, beta, order):
    rng = np.random.default_rng(M + N + K)
    A, B, C0 = rng.standard_normal((K, M)), rng.standard_normal((K, N)), rng.standard_normal((M, N))
    dA, lA, hA = ((K, M), (-1, 1), A) if order == "km" else ((M, K), (1, -1), A.T)
    p = ctx.plan_dense(dA, lA, (K, N), (-1, 2), (M, N), (1, 2))
    assert p.info["tile"] == 5
    a, b, c = dev.put(hA), dev.put(B), dev.put(C0)
    p.execute(a.data_ptr(), b.data_ptr(), c.data_ptr(), 2.0, beta)
    got = dev.get(c, (M, N))
    bound = (K + 3) * EPS * (2 * np.abs(A.T) @ np.abs(B) + np.abs(beta * C0))
    assert np.all(np.abs(got - (2.0 * A.T @ B + beta * C0)) <= bound)


@pytest.mark.parametrize("dims", [[(300, 9, 20), (300, 9, 7)], [(257, 17, 1), (257, 17, 64), (257, 17, 21)]])
def test_skinny_tasks_of_one_block(ctx, dev, dims):
    rng = np.random.default_rng(len(dims))
    M, N = dims[0][:2]
    A = [rng.standard_normal((k, M)) for _, _, k in dims]
    B = [rng.standard_normal((k, N)) for _, _, k in dims]
    offs, blkA, blkB, a, b = [], [], [], 0, 0
    for _, _, k in dims:
        offs += [a, b, 0]
        blkA += [k, M]
        blkB += [k, N]
        a, b = a + k * M, b + k * N
    p = ctx.plan_qn((-1, 1), (-1, 2), (1, 2), offs, blkA, blkB)
    assert p.info["tile"] == 5
    c = dev.empty(M * N)
    Ad = dev.put(np.concatenate([x.ravel(order="F") for x in A]))
    Bd = dev.put(np.concatenate([x.ravel(order="F") for x in B]))
    p.execute(Ad.data_ptr(), Bd.data_ptr(), c.data_ptr())
    ref = sum(x.T @ y for x, y in zip(A, B))
    K = sum(k for _, _, k in dims)
    assert np.all(np.abs(dev.get(c, (M, N)) - ref) <= (K + 3) * EPS * sum(np.abs(x.T) @ np.abs(y) for x, y in zip(A, B)))


@pytest.mark.parametrize("N", [9, 16, 17, 32])
@pytest.mark.parametrize("Ks", [[1], [4], [5], [12], [13], [20], [21], [24], [25], [32], [33], [1, 4], [3, 5, 12], [13, 2], [64, 1]])
def test_skinny_slots(ctx, dev, Ks, N):
    """Remainders of k in one, three and five slots of four, one task and several."""
    rng = np.random.default_rng(sum(Ks) + N)
    M = 321
    A, B = [rng.standard_normal((k, M)) for k in Ks], [rng.standard_normal((k, N)) for k in Ks]
    offs, blkA, blkB, a, b = [], [], [], 0, 0
    for k in Ks:
        offs += [a, b, 0]
        blkA += [k, M]
        blkB += [k, N]
        a, b = a + k * M, b + k * N
    p = ctx.plan_qn((-1, 1), (-1, 2), (1, 2), offs, blkA, blkB)
    assert p.info["tile"] == 5
    Ad, Bd, c = dev.put(np.concatenate([x.ravel(order="F") for x in A])), dev.put(np.concatenate([x.ravel(order="F") for x in B])), dev.empty(M * N)
    p.execute(Ad.data_ptr(), Bd.data_ptr(), c.data_ptr())
    ref = sum(x.T @ y for x, y in zip(A, B))
    bound = (sum(Ks) + 3) * EPS * sum(np.abs(x.T) @ np.abs(y) for x, y in zip(A, B))
    assert np.all(np.abs(dev.get(c, (M, N)) - ref) <= bound)
