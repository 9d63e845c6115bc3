"""The FP32 and BF16x3 small-block kernels either side of the k (24) up to
which lanes walk the rows in every layout: the layout does not enter the sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = {"f32": np.finfo(np.float32).eps, "bf16x3": 2.0**-14}


def _run(ctx, dev, shapes, aorder, border, prec):
    rng = np.random.default_rng(len(shapes))
    A, B, offs, bA, bB, c0, refs = [], [], [], [], [], 0, []
    na = nb = 0
    for (M, N), Ks in shapes:
        ref, bound = np.zeros((M, N)), np.zeros((M, N))
        for K in Ks:
            a, b = rng.standard_normal((M, K)), rng.standard_normal((K, N))
            offs += [na, nb, c0]
            bA += [K, M] if aorder == "km" else [M, K]
            bB += [K, N] if border == "kn" else [N, K]
            A.append((a.T if aorder == "km" else a).ravel(order="F"))
            B.append((b if border == "kn" else b.T).ravel(order="F"))
            na, nb = na + M * K, nb + K * N
            ref += a @ b
            bound += np.abs(a) @ np.abs(b)
        refs.append((c0, ref, bound, sum(Ks)))
        c0 += M * N
    p = ctx.plan_qn((-1, 1) if aorder == "km" else (1, -1), (-1, 2) if border == "kn" else (2, -1), (1, 2), offs, bA, bB,
                    prec)
    assert p.info["tile"] == 10
    Ad, Bd, C = dev.put(np.concatenate(A)), dev.put(np.concatenate(B)), dev.empty(c0)
    p.execute(Ad.data_ptr(), Bd.data_ptr(), C.data_ptr(), 1.5)
    got = dev.get(C, (c0,))
    for o, ref, bound, K in refs:
        x = got[o:o + ref.size].reshape(ref.shape, order="F")
        assert np.all(np.abs(x - 1.5 * ref) <= (K + 3) * EPS[prec] * 1.5 * bound)
    return got


@pytest.mark.parametrize("prec", ["f32", "bf16x3"])
@pytest.mark.parametrize("shapes", [
    [((1, 1), [1])], [((65, 33), [8, 1, 3])], [((63, 31), [24, 5])], [((61, 30), [25, 24])], [((64, 32), [65, 2])], [((60, 15), [1, 8])] * 23,
    [((40, 37), [64] * 7), ((5, 9), [3])], [((90, 80), [64] * 40)] * 2, [((90, 90), [3000])],  # split over units
], ids=range(9))
def test_small_blocks_reduced(ctx, dev, shapes, prec):
    got = [_run(ctx, dev, shapes, a, b, prec) for a in ("km", "mk") for b in ("kn", "nk")]
    assert all(np.array_equal(got[0], x) for x in got[1:])
