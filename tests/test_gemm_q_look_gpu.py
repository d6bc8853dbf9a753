"""Products of a quantized W with many columns of x: outputs that the bf16 terms
of x cannot form (infinities, sums beyond the largest float, x below what the
terms hold) are formed from f32 products, at a bounded cost."""
import pytest
import torch

import vortx_amd as vx
from tests.helpers import note

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BLOCK = {vx.VX_Q4_0: (32, 18), vx.VX_Q8_0: (32, 34), vx.VX_Q4_K: (256, 144)}
QTYPES = pytest.mark.parametrize("qtype", list(BLOCK), ids=["q4_0", "q8_0", "q4_k"])


def _weights(qgemv, qtype, M, K, seed, zero=0):
    """A quantized normal matrix (its first `zero` columns zeros), and its values."""
    qk, bb = BLOCK[qtype]
    g = torch.Generator(device=DEV).manual_seed(seed)
    v = torch.randn(M, K, device=DEV, generator=g) * K ** -0.5
    v[:, :zero] = 0.0
    w = vx.QWeight(torch.empty(M * (K // qk) * bb, dtype=torch.uint8, device=DEV), qtype, M, K)
    qgemv.quantize(w, v)
    wd = torch.empty(M, K, device=DEV)
    qgemv.dequantize(wd, w)
    return w, wd


def _x(B, K, seed):
    return torch.randn(B, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed))


def _bound(x, wd, exact_x):
    """|error|: a few f32 roundings per 32-block of the magnitudes added (at most
    3 times the block's largest weight per element of x), and x to 2^-16."""
    K = x.shape[1]
    mag = 3.0 * wd.double().abs().view(-1, K // 32, 32).amax(-1).repeat_interleave(32, 1)
    return ((K / 32 + 48) * 2.0 ** -24 + (0.0 if exact_x else 2.0 ** -16)) * (x.double().abs() @ mag.t())


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


@QTYPES
@pytest.mark.parametrize("M,B", [(2000, 40), (2300, 1901)])
def test_cost_of_non_finite_x(qgemv, qtype, M, B):
    """A NaN or an infinity in every column, or only zeros: the outputs of the f32 products,
    and a bounded time (measured 1.4 times an ordinary x's with NaNs or zeros, 3 to 6
    times with infinities; forming each output in one lane took 22 times and more)."""
    K = 2048
    note(f"gemm_q cost of non-finite {qtype} {M} B={B}")
    w, wd = _weights(qgemv, qtype, M, K, 1)
    x = _x(B, K, 2)
    y = torch.empty(B, M, device=DEV)
    call = lambda v: qgemv.dispatch(y.t(), w, v.t(), x_f32=True)  # noqa: E731
    base = _us(lambda: call(x))
    for bad in (float("nan"), float("inf"), 0.0):
        xb = x.clone() if bad else torch.zeros_like(x)
        xb[torch.arange(B), torch.arange(B) % K] = bad
        us = _us(lambda: call(xb))
        note(f"  {bad}: {us:.0f} us, {base:.0f} without")
        want = xb.double() @ wd.double().t()
        assert torch.equal(y.isnan(), want.isnan())
        inf = want.isinf()
        assert torch.equal(y[inf].double(), want[inf])
        assert us < 12 * base + 50, f"{bad}: {us:.0f} us, {base:.0f} without"


@QTYPES
@pytest.mark.parametrize("M,B", [(300, 9), (2300, 1901)])
@pytest.mark.parametrize("e", [-116, -122, -131])
def test_small_x_keeps_its_bits(qgemv, qtype, M, B, e):
    """x kept in f32 far below one (its third terms would fall below bf16's
    smallest number, 2^-133): whole columns, and elements that are all that
    counts beside larger ones whose weights are zeros."""
    K = 512
    note(f"gemm_q small x {qtype} {M} B={B} 2^{e}")
    w, wd = _weights(qgemv, qtype, M, K, 3, zero=256)
    x = _x(B, K, 4)
    x[::2] = torch.ldexp(x[::2], torch.tensor(e, device=DEV))
    x[1, 256:] = torch.ldexp(x[1, 256:], torch.tensor(e, device=DEV))
    x[3, 300:] = 0.0
    y, y2 = torch.empty(B, M, device=DEV), torch.empty(M, B, device=DEV)
    qgemv.dispatch(y.t(), w, x.t(), x_f32=True)
    qgemv.dispatch(y2, w, x.t().contiguous(), x_f32=True)
    err = (y.double() - x.double() @ wd.double().t()).abs()
    bound = _bound(x, wd, True) + K * 2.0 ** -149
    assert (err <= bound).all(), f"{float((err / bound).max())} of the bound"
    assert torch.equal(y, y2.t())


@QTYPES
@pytest.mark.parametrize("M,B", [(300, 40), (2300, 1901)])
def test_large_x_with_a_workspace(qgemv, qtype, M, B):
    """x around 1e37 with a workspace: a block's whole-number sum (up to 32 x 127
    times x) is beyond the largest float, the result is not."""
    K = 512
    note(f"gemm_q large x {qtype} {M} B={B}")
    w, wd = _weights(qgemv, qtype, M, K, 5)
    x = _x(B, K, 6).clamp_(-3, 3)
    x[::2] *= 1e37
    y = torch.empty(B, M, device=DEV)
    qgemv.dispatch(y.t(), w, x.t(), workspace=vx.QuantGemv.workspace(w, B))
    err = (y.double() - x.double() @ wd.double().t()).abs()
    bound = _bound(x, wd, False)
    assert (err <= bound).all(), f"{float((err / bound).max())} of the bound"
