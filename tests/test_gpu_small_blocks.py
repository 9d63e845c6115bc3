"""The FP64 small-block path at the edges of its units (16, 32 and 64 rows,
16 and 32 columns), k loads (16) and wave sharing (tasks against waves), for
every operand layout, alone and split over units."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _run(ctx, dev, shapes, aorder, border, alpha=1.5):
    """C (M x N) = alpha sum over tasks A_t B_t, K_t each; several C blocks."""
    rng = np.random.default_rng(len(shapes) + sum(map(sum, (s[1] for s in shapes))))
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
    p = ctx.plan_qn((-1, 1) if aorder == "km" else (1, -1), (-1, 2) if border == "kn" else (2, -1), (1, 2), offs, bA, bB)
    assert p.info["tile"] == 10
    Ad, Bd, C = dev.put(np.concatenate(A)), dev.put(np.concatenate(B)), dev.empty(c0)
    p.execute(Ad.data_ptr(), Bd.data_ptr(), C.data_ptr(), alpha)
    got = dev.get(C, (c0,))
    for o, ref, bound, K in refs:
        x = got[o:o + ref.size].reshape(ref.shape, order="F")
        assert np.all(np.abs(x - alpha * ref) <= (K + 3) * EPS * alpha * bound)


@pytest.mark.parametrize("aorder", ["km", "mk"])
@pytest.mark.parametrize("border", ["kn", "nk"])
@pytest.mark.parametrize("shapes", [
    [((1, 1), [1])], [((16, 16), [16])], [((17, 15), [17]), ((15, 17), [15])],
    [((33, 32), [64, 1, 3])], [((31, 33), [5] * 9)], [((64, 65), [40] * 3), ((65, 31), [7] * 20)],
    [((128, 64), [160])], [((100, 70), [16, 32, 48, 64, 80])],
    [((40, 37), [23, 11])] * 300, [((70, 40), [33])] * 150,  # units of 64 and of 32 rows
    [((30, 30), [50] * 60)], [((90, 80), [64] * 40)] * 2,    # split over units
], ids=range(12))
def test_small_blocks(ctx, dev, monkeypatch, shapes, aorder, border):
    monkeypatch.setenv("ITX_FORCE_TILE", "10")  # also where the 32 x 32 tile is the default
    _run(ctx, dev, shapes, aorder, border)
