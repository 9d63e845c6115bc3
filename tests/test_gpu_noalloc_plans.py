"""itx_contract_qn_noalloc runs the plan of itx_contract_qn -- finer units for
few blocks, k split over units -- and so gives its bits, wherever the scratch
array holds that plan; where it does not, a plan with less in it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _both(ctx, M, N, Ks, order, prec):
    import torch

    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + N + sum(Ks))
    offs, bA, bB, a, b, ref = [], [], [], [], [], 0.0
    na = nb = 0
    for K in Ks:
        x = torch.randn(M, K, dtype=torch.float64, device=dev, generator=g)
        y = torch.randn(N, K, dtype=torch.float64, device=dev, generator=g)
        offs += [na, nb, 0]
        bA += [K, M] if order == "k" else [M, K]
        bB += [K, N] if order == "k" else [N, K]
        a.append((x if order == "k" else x.t()).reshape(-1))
        b.append((y if order == "k" else y.t()).reshape(-1))
        na, nb = na + M * K, nb + K * N
        if len(Ks) * K < 100000:
            ref = ref + y @ x.t()  # column-major C
        else:
            ref = sum(y[:, i:i + 4096] @ x[:, i:i + 4096].t() for i in range(0, K, 4096))
    A, B = torch.cat(a), torch.cat(b)
    del a, b
    lab = ((-1, 1), (-1, 2)) if order == "k" else ((1, -1), (2, -1))
    out = []
    for noalloc in (False, True):
        C = torch.full((M * N,), float("nan"), dtype=torch.float64, device=dev)
        ctx.contract_qn(A.data_ptr(), lab[0], B.data_ptr(), lab[1], C.data_ptr(), (1, 2), offs, bA, bB, 1.0, prec,
                        noalloc=noalloc)
        out.append(C)
    torch.cuda.synchronize()
    return out[0], out[1], ref.reshape(-1)


@pytest.mark.parametrize("order", ["k", "m"])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16x3"])
@pytest.mark.parametrize("M,N,Ks", [(60, 40, [400]), (128, 32, [160]), (64, 32, [17]), (7, 5, [2500]), (60, 40, [90] * 9),
                                    (200, 200, [2000]), (65, 130, [5000]), (300, 200, [500]), (255, 253, [129])])
def test_noalloc_bits(ctx, M, N, Ks, prec, order):
    ref, got, _ = _both(ctx, M, N, Ks, order, prec)
    assert (ref == got).all()


@pytest.mark.parametrize("M,N,K", [(200, 199, 1060000), (90, 120, 1800000)])
def test_noalloc_less_than_the_ordinary_plan(ctx, M, N, K):
    """Offset tables of more than half the 32 MiB scratch: no room for the partial tiles as well."""
    a, b, ref = _both(ctx, M, N, [K], "m", "f64")
    bound = (K + 70) * EPS * 2.0 * K  # |x| |y| sums to 2 K / pi on average
    assert float((a - ref).abs().max()) <= bound and float((b - ref).abs().max()) <= bound
