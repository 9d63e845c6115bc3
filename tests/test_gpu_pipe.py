"""The FP64 pipelined tiles (64 x 64 and 128 x 128) at the edges of tiles and
k stages (16, five and more for the steady state), for every operand layout
and alignment, several tasks per block, split over k, and as chosen by
default against the same sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
SHAPES = [
    [((1, 1), [1])], [((64, 64), [16])], [((65, 63), [17, 1])], [((63, 129), [96])], [((128, 128), [80])],
    [((127, 130), [95, 33, 2])], [((50, 200), [47] * 3), ((200, 50), [64])],
    [((30, 70), [96])] * 40, [((20, 90), [5, 31])] * 9,  # XCD lists of several blocks
    [((70, 60), [129])], [((150, 40), [1000])], [((64, 65), [4097])],  # split over k
]


def _run(ctx, dev, shapes, aorder, border, tile, odd, alpha=1.5, beta=0.0, prec="f64"):
    """C (M x N) = alpha sum over tasks A_t B_t (+ beta C); several C blocks."""
    # BF16x3: both terms of an operand hold 16 bits, and lo * lo is dropped
    eps = {"f64": EPS, "f32": np.finfo(np.float32).eps, "bf16x3": 2.0**-14}[prec]
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
    p = ctx.plan_qn((-1, 1) if aorder == "km" else (1, -1), (-1, 2) if border == "kn" else (2, -1), (1, 2), offs, bA, bB, prec=prec)
    assert tile is None or p.info["tile"] == tile
    pad = np.zeros(odd)  # an operand 8 bytes off its allocation: single loads
    c = rng.standard_normal(c0)
    Ad, Bd, C = dev.put(np.concatenate([pad, *A])), dev.put(np.concatenate([pad, *B])), dev.put(c)
    p.execute(Ad.data_ptr() + 8 * odd, Bd.data_ptr() + 8 * odd, C.data_ptr(), alpha, beta)
    got = dev.get(C, (c0,))
    for o, ref, bound, K in refs:
        x, y = (v[o:o + ref.size].reshape(ref.shape, order="F") for v in (got, c))
        assert np.all(np.abs(x - alpha * ref - beta * y) <= (K + 70) * eps * (alpha * bound + abs(beta * y)))
    return got


@pytest.mark.parametrize("tile", [16, 17, None])
@pytest.mark.parametrize("aorder,border,odd", [("km", "kn", 0), ("km", "kn", 1), ("km", "nk", 0), ("mk", "kn", 0), ("mk", "nk", 1)])
@pytest.mark.parametrize("shapes", SHAPES, ids=range(len(SHAPES)))
def test_pipe(ctx, dev, monkeypatch, shapes, aorder, border, odd, tile):
    if tile is not None:
        monkeypatch.setenv("ITX_FORCE_TILE", str(tile))
    _run(ctx, dev, shapes, aorder, border, tile, odd)


@pytest.mark.parametrize("tile", [16, 17])
def test_pipe_beta(ctx, dev, monkeypatch, tile):
    monkeypatch.setenv("ITX_FORCE_TILE", str(tile))
    _run(ctx, dev, [((70, 60), [129])], "km", "kn", tile, 0, beta=-0.5)


@pytest.mark.parametrize("shapes", [
    [((300, 3), [3, 3, 1]), ((300, 2), [3, 3]), ((700, 3), [2, 3]), ((4, 3), [3])] * 30,  # narrow, tiny
    [((600, 20), [30, 7])] * 12,                                                          # narrow
], ids=["tiny", "narrow"])
def test_narrow_lists(ctx, dev, shapes):
    _run(ctx, dev, shapes, "mk", "kn", 5, 0)


@pytest.mark.parametrize("aorder,border,odd", [("km", "kn", 0), ("km", "kn", 1), ("km", "nk", 0), ("mk", "kn", 0), ("mk", "nk", 1)])
@pytest.mark.parametrize("shapes", SHAPES, ids=range(len(SHAPES)))
@pytest.mark.parametrize("prec,tiles", [("f32", (4, 16, 17, 18)), ("bf16x3", (4, 16, 17))])
def test_pipe_same_bits(ctx, dev, monkeypatch, shapes, aorder, border, odd, prec, tiles):
    """The FP32 and BF16x3 tiles sum in one order: the same bits from all of them."""
    got = []
    for tile in tiles:
        monkeypatch.setenv("ITX_FORCE_TILE", str(tile))
        got.append(_run(ctx, dev, shapes, aorder, border, tile, odd, beta=0.25, prec=prec))
    for x in got[1:]:
        assert np.array_equal(got[0], x)


@pytest.mark.parametrize("tile", [16, 17])
@pytest.mark.parametrize("M,N,K", [(65, 63, 32), (64, 70, 96), (130, 127, 35), (1, 1, 1)])
def test_pipe_split_words(ctx, dev, monkeypatch, M, N, K, tile):
    """Pre-split operands give the bits of the FP64 operands."""
    monkeypatch.setenv("ITX_FORCE_TILE", str(tile))
    rng = np.random.default_rng(M + N + K)
    ops = [dev.put(rng.standard_normal(K * x)) for x in (M, N)]
    words = [dev.empty(x.numel()) for x in ops]
    for x, w in zip(ops, words):
        ctx.split_bf16(x.data_ptr(), w.data_ptr(), x.numel())
    p = ctx.plan_qn((-1, 1), (-1, 2), (1, 2), [0, 0, 0], [K, M], [K, N], prec="bf16x3")
    C = dev.empty(M * N)
    p.execute(ops[0].data_ptr(), ops[1].data_ptr(), C.data_ptr())
    want = dev.get(C, (M * N,)).copy()
    if K == 1:  # no contracted index: refused as before
        with pytest.raises(Exception):
            p.set_split(True)
        return
    p.set_split(True)
    p.execute(words[0].data_ptr(), words[1].data_ptr(), C.data_ptr())
    assert np.array_equal(want, dev.get(C, (M * N,)))
