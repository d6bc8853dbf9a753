"""The f32 GEMM on the bf16 matrix cores (operands as three bf16 terms each) at
the edges of its tiles and its K split, against float64.

Error bound, elementwise: six of the nine products of terms are formed, the
others are below 2^-24 of |a b| together; every product is exact and is added
in f32, six additions per 16 elements of K at most (and a few at the end):
(6 K / 16 + 16) roundings of 2^-24 of sum |a b| at most, in practice their
square root."""
import numpy as np
import pytest
import torch

import vortx_amd as vx
from tests.helpers import note
from vortx_amd import synthetic as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _bits(t):
    return t.contiguous().view(torch.int32)


def _check(c, a, b, K, what, alpha=1.0, beta=0.0, c0=None):
    a, b = a.double(), b.double()
    ref = alpha * (a @ b) + (beta * c0.double() if beta else 0.0)
    bound = abs(alpha) * ((6 * K / 16 + 16) * 2.0 ** -24) * (a.abs() @ b.abs()) + 2.0 ** -22 * ref.abs() + 1e-37
    if beta:
        bound = bound + 2.0 ** -22 * (beta * c0.double()).abs()
    err = (c.double() - ref).abs()
    assert bool((err <= bound).all()), f"{what}: {float((err / bound).max())} of the bound"


# (M, N, K, batch): around 32 (the K split), 64, 128 and 256 (the tiles), K
# around 32, 64 and 256 (stages, chunks of a wave). Kernels on 256 CUs
# (tests/test_kernel_choice.py): k16 up to 100 x 70, then 64 x 64 with short
# stages, twice, 128 x 128, 256 x 128; 64 x 64 with long stages (an odd and an
# even number of them, with and without a tail), ks (with a tail, whole, a tail
# alone on a wave), 256 x 128 twice
SHAPES = [(32, 32, 64, 1), (31, 33, 31, 1), (33, 95, 257, 2), (1, 64, 4097, 1), (64, 1, 65, 3), (100, 70, 8, 1),
          (1000, 1030, 161, 1), (1111, 1200, 192, 1), (2100, 1900, 170, 1), (1300, 1100, 130, 12),
          (970, 1000, 673, 1), (1000, 1001, 1023, 1), (1000, 1003, 768, 1), (300, 517, 609, 1), (513, 301, 768, 1), (300, 517, 257, 1),
          (4000, 4011, 500, 1), (2048, 4096, 333, 1)]


@pytest.mark.parametrize("M,N,K,batch", SHAPES, ids=[f"{m}x{n}x{k}-{b}" for m, n, k, b in SHAPES])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)],
                         ids=["ab", "abT", "aTb", "aTbT"])
def test_gemm_bf(gemm, M, N, K, batch, ta, tb):
    note(f"gemm_bf {M}x{N}x{K} batch {batch} ta={ta} tb={tb}")
    a = S.uniform((batch, K, M) if ta else (batch, M, K), M, DEV)
    b = S.uniform((batch, N, K) if tb else (batch, K, N), N + 1, DEV)
    a, b = a.transpose(1, 2) if ta else a, b.transpose(1, 2) if tb else b
    c = torch.full((batch, M, N), float("nan"), device=DEV)
    gemm.dispatch_tiled(c, a, b)
    torch.cuda.synchronize()
    _check(c, a, b, K, "plain")
    c0 = S.uniform((batch, M, N), 7, DEV)
    c1 = c0.clone()
    gemm.dispatch_ex(c1, a, b, alpha=-0.5, beta=2.0)
    torch.cuda.synchronize()
    if N > 1 and (M >= 32 or N >= 32):  # (other routes otherwise)
        _check(c1, a, b, K, "alpha, beta", -0.5, 2.0, c0)


# small: 64 x 64 with long stages, short ones, short ones
@pytest.mark.parametrize("M,N,K", [(970, 1000, 673), (1500, 1333, 200), (2048, 2048, 160)])
def test_tile_shapes_give_the_same_bits(gemm, M, N, K):
    note(f"gemm_bf tiles {M}x{N}x{K}")
    a, b = S.uniform((M, K), 1, DEV), S.uniform((N, K), 2, DEV).t()
    out = []
    for tile in ("auto", "narrow", "wide", "small"):
        out.append(torch.full((M, N), float("nan"), device=DEV))
        gemm.dispatch_ex(out[-1], a, b, tile=tile)
    torch.cuda.synchronize()
    _check(out[0], a, b, K, "auto")
    for c in out[1:]:
        assert torch.equal(_bits(c), _bits(out[0]))


# k16, ks, 64 x 64 with short and long stages, 128 x 128, 256 x 128
KERNELS = pytest.mark.parametrize("M,N,K", [(70, 80, 300), (300, 517, 600), (1200, 1100, 300), (970, 1000, 673), (2100, 1900, 170),
                                            (4000, 4011, 500)], ids=["k16", "ks", "s", "s2", "n", "w"])


@KERNELS
def test_non_finite_operands(gemm, M, N, K):
    """Infinities keep their sign, NaNs stay where they belong, and the largest
    finite floats are not taken for infinities."""
    note(f"gemm_bf non-finite {M}x{N}x{K}")
    a, b = S.uniform((M, K), 3, DEV) + 2.0, S.uniform((K, N), 4, DEV)
    a[3, 17], a[5, K - 1], b[min(200, K - 2), 9] = float("inf"), float("nan"), -float("inf")
    a[7, :], b[0, 11] = 0.0, torch.finfo(torch.float32).max
    a[8, :] = 0.0
    a[8, 0] = 0.5
    c = torch.full((M, N), 1.0, device=DEV)
    gemm.dispatch_tiled(c, a, b)
    torch.cuda.synchronize()
    an, bn = a.cpu().numpy(), b.cpu().numpy()
    ref = np.zeros((12, N), np.float32)  # one product at a time in f32
    with np.errstate(all="ignore"):
        for k in range(K):
            ref += an[:12, k, None] * bn[k]
    got = c[:12].cpu().numpy()
    assert bool((np.isnan(got) == np.isnan(ref)).all())
    inf = np.isinf(ref)
    assert bool((got[inf] == ref[inf]).all())
    assert got[8, 11] == np.float32(0.5) * np.finfo(np.float32).max
    assert torch.isfinite(c[12:, 12:]).all()


@KERNELS
@pytest.mark.parametrize("ea,eb", [(-120, 60), (-60, -50), (-100, -30), (70, 40)])
def test_far_from_one(gemm, M, N, K, ea, eb):
    """Operands whose smaller terms would fall below bf16's or f32's smallest
    numbers (whole matrices, and single rows and columns among others of
    ordinary size) lose nothing."""
    note(f"gemm_bf scales 2^{ea} 2^{eb}")
    a, b = S.uniform((M, K), 5, DEV), S.uniform((K, N), 6, DEV)
    for rows in (slice(None), slice(5, 6)):
        aa, bb = a.clone(), b.clone()
        aa[rows] = torch.ldexp(a[rows], torch.tensor(ea, device=DEV))
        bb[:, rows] = torch.ldexp(b[:, rows], torch.tensor(eb, device=DEV))
        c = torch.full((M, N), float("nan"), device=DEV)
        gemm.dispatch_tiled(c, aa, bb)
        torch.cuda.synchronize()
        ref = aa.double() @ bb.double()
        mag = aa.double().abs() @ bb.double().abs()
        err = (c.double() - ref).abs()
        assert bool((err <= (K + 32) * 2.0 ** -24 * mag + K * 2.0 ** -126).all()), float((err / mag).max())
