"""f32 GEMM: outputs that the bf16 terms of the operands cannot form (infinities,
elements below what three terms hold) are formed from f32 products, in every
kernel that works on terms."""
import pytest
import torch

from tests.helpers import note
from vortx_amd import synthetic as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# 16 x 16 and 32 x 32 tiles with K split; 64 x 64 tiles with short and long
# stages; 128 x 128; 256 x 128
SHAPES = pytest.mark.parametrize("M,N,K", [(70, 80, 300), (300, 517, 600), (1200, 1100, 300), (970, 1000, 673),
                                           (2100, 1900, 170), (4000, 4011, 500)])
MODES = pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)],
                                ids=["ab", "abT", "aTb", "aTbT"])


def _run(gemm, a, b, ta, tb):
    """a b with the operands stored transposed or not."""
    a = a.t().contiguous().t() if ta else a
    b = b.t().contiguous().t() if tb else b
    c = torch.full((a.shape[0], b.shape[1]), float("nan"), device=DEV)
    gemm.dispatch_tiled(c, a, b)
    return c


@MODES
@SHAPES
def test_small_elements_beside_large_ones(gemm, M, N, K, ta, tb):
    """Elements around 2^-120 are all that counts where the larger ones beside
    them meet zeros: to f32's own bound, elementwise."""
    note(f"gemm_bf mixed magnitudes {M}x{N}x{K} ta={ta} tb={tb}")
    a, b = S.uniform((M, K), 1, DEV), S.uniform((K, N), 2, DEV)
    a[5, 3:] = torch.ldexp(a[5, 3:], torch.tensor(-120, device=DEV))    # a row: large for k < 3, where some columns are 0
    a[11] = torch.ldexp(a[11], torch.tensor(-126, device=DEV))
    a[9, 7:] = torch.ldexp(a[9, 7:], torch.tensor(-140, device=DEV))
    b[:7, ::3] = 0.0
    b[:, 4::9] = torch.ldexp(b[:, 4::9], torch.tensor(100, device=DEV))
    b[20:, 7] = torch.ldexp(b[20:, 7], torch.tensor(-122, device=DEV))  # a column, the same way
    a[20:30, :20] = 0.0
    a[30:40] = torch.ldexp(a[30:40], torch.tensor(-75, device=DEV))     # products below 2^-126
    b[:, 40:45] = torch.ldexp(b[:, 40:45], torch.tensor(-60, device=DEV))
    c = _run(gemm, a, b, ta, tb)
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    err, bound = (c.double() - ref).abs(), (K + 32) * 2.0 ** -24 * mag + K * 2.0 ** -149
    assert bool((err <= bound).all()), f"{float((err / bound).max())} of the bound"


def _us(f):
    f()
    best = float("inf")
    for _ in range(5):
        t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        t0.record()
        f()
        t1.record()
        torch.cuda.synchronize()
        best = min(best, t0.elapsed_time(t1) * 1e3)
    return best


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)], ids=["ab", "aTbT"])
@pytest.mark.parametrize("M,N,K", [(16, 1600, 4096), (300, 517, 4096), (1200, 1100, 1000), (970, 1000, 2000), (2100, 1900, 1000),
                                   (4000, 4011, 1000)])
def test_cost_of_non_finite_and_small(gemm, M, N, K, ta, tb):
    """A NaN or an infinity in every row, or products far below one: what f32
    products give, in a bounded time (measured up to 5.5 times an ordinary
    call's; forming each output in one lane took 20 times and more)."""
    note(f"gemm_bf cost {M}x{N}x{K} ta={ta} tb={tb}")
    a, b = S.uniform((M, K), 1, DEV) + 2.0, S.uniform((K, N), 2, DEV)
    a = a.t().contiguous().t() if ta else a
    b = b.t().contiguous().t() if tb else b
    c = torch.empty((M, N), device=DEV)
    base = _us(lambda: gemm.dispatch_tiled(c, a, b))
    rows = torch.arange(M, device=DEV)
    for what in ("nan", "inf", "1e-13", "1e-20"):
        aa, bb = (a * float(what), b * float(what)) if what[0] == "1" else (a.clone(), b)
        if what[0] != "1":
            aa[rows, rows % K] = float(what)
        us = _us(lambda: gemm.dispatch_tiled(c, aa, bb))
        note(f"  {what}: {us:.0f} us, {base:.0f} without")
        ref = aa.double() @ bb.double()
        if what[0] == "1":
            bound = (K + 32) * 2.0 ** -24 * (aa.double().abs() @ bb.double().abs()) + K * 2.0 ** -149
            assert bool(((c.double() - ref).abs() <= bound).all()), what
        else:
            assert torch.equal(c.isnan(), ref.isnan()) and torch.equal(c[ref.isinf()].double(), ref[ref.isinf()])
        assert us < (2 if what == "1e-13" else 8) * base + 50, f"{what}: {us:.0f} us, {base:.0f} without"
