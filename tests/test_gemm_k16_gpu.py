"""f32 GEMM in 16 x 16 tiles with K split over a workgroup (few outputs, long K)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(n, M, N, K, ta, tb, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn((n, K, M) if ta else (n, M, K), device="cuda", generator=g)
    b = torch.randn((n, N, K) if tb else (n, K, N), device="cuda", generator=g)
    return (a.transpose(1, 2) if ta else a), (b.transpose(1, 2) if tb else b)


def _check(got, a, b, alpha=1.0, beta=0.0, c0=None):
    """Dropped products are below 2^-24 of each |a b|, the f32 sums round once
    per addition: at most K + 64 roundings of sum |a||b|, plus the epilogue's."""
    K = a.shape[-1]
    want = alpha * (a.double() @ b.double())
    mag = abs(alpha) * (a.double().abs() @ b.double().abs())
    if beta:
        want, mag = want + beta * c0.double(), mag + abs(beta) * c0.double().abs()
    assert ((got.double() - want).abs() <= (K + 64) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("n,M,N,K", [(1, 32, 32, 1), (1, 33, 1, 31), (1, 33, 47, 33), (1, 1, 1000, 256), (2, 17, 49, 257),
                                     (1, 15, 4111, 2100), (1, 16, 1600, 4096), (3, 96, 65, 1031), (1, 40, 100, 7999)])
def test_sizes_and_strides(gemm, n, M, N, K, ta, tb):
    a, b = _operands(n, M, N, K, ta, tb, M + K)
    out = torch.full((n, M, N), float("nan"), device="cuda")
    gemm.dispatch(out, a, b)
    _check(out, a, b)
    c0 = torch.randn(n, N, M, device="cuda").transpose(1, 2)
    out = c0.clone()
    gemm.dispatch_ex(out, a, b, alpha=0.5, beta=-2.0)
    _check(out, a, b, 0.5, -2.0, c0)


def test_extreme_values(gemm):
    """Infinities, NaN, products below and above what the split holds: the
    outputs a plain sequential f32 sum gives, within its own bound."""
    a, b = _operands(1, 40, 50, 600, False, True, 3)
    a[0, 3, 100] = float("inf")
    a[0, 5, 7] = float("nan")
    b[0, 9, 20] = -float("inf")
    a[0, 8] *= 1e-30
    b[0, :, 11] *= 1e-12
    a[0, 10] = 3.402e38
    b[0, :, 13] = 0.0
    a[0, 12] *= 1e-42
    out = torch.empty(1, 40, 50, device="cuda")
    gemm.dispatch(out, a, b)
    want = a.double() @ b.double()
    mag = a.double().abs() @ b.double().abs()
    fin = torch.isfinite(mag) & (mag < 3.4e38)
    err = (out.double() - want).abs()
    assert (err[fin] <= (600 + 64) * 2.0 ** -24 * mag[fin] + 600 * 2.0 ** -149).all()
    # outputs that are not finite: redone in f32 from the first k to the last
    seq = torch.zeros(40, 50)
    ac, bc = a[0].cpu(), b[0].cpu()
    for k in range(600):
        seq = torch.addcmul(seq, ac[:, k:k + 1].expand(40, 50), bc[k:k + 1].expand(40, 50))
    got = out[0].cpu()
    assert torch.isnan(got)[torch.isnan(seq)].all()
    inf = torch.isinf(seq)
    assert inf.any() and (got[inf] == seq[inf]).all()
