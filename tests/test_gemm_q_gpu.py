"""Products of a quantized W with many columns of x (the bf16 matrix-core
kernels: x as two bf16 terms with a workspace and more than 16 columns, as
three, exactly, with VX_GEMV_X_F32 or without a workspace and more than four),
at the edges of their tiles, against float64.

Error bounds, elementwise: each 32-block's sum is formed from exact products
in f32 and the blocks are added in f32, so at most (K / 32 + 48) roundings of
2^-24 of the magnitudes added; those are at most 3 max|W_block| |x| per
element (nibbles are used unbiased or centred, their offset added per block).
Two terms of x are off by at most 2^-16 |x|."""
import numpy as np
import pytest
import torch

import vortx_amd as vx
from oracle import oracle as O
from tests.helpers import note
from vortx_amd import synthetic as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
QTYPES = [vx.VX_Q4_0, vx.VX_Q8_0, vx.VX_Q4_K]
QN = {vx.VX_Q4_0: "q4_0", vx.VX_Q8_0: "q8_0", vx.VX_Q4_K: "q4_k"}


def _reference(qtype, w, M, K, x):
    """(W x in float64, the sum of the magnitudes that the kernels add), both [B, M]."""
    wd = O.dequant(qtype, w.cpu().numpy(), M, K).astype(np.float64)
    mag = np.repeat(3.0 * np.abs(wd).reshape(M, K // 32, 32).max(-1), 32, axis=1)
    x = x.cpu().numpy().astype(np.float64)
    return x @ wd.T, np.abs(x) @ mag.T


def _check(y, ref, mag, K, exact_x, what):
    err = np.abs(y.cpu().numpy().astype(np.float64) - ref)
    bound = ((K / 32 + 48) * 2.0 ** -24 + (0.0 if exact_x else 2.0 ** -16)) * mag + 1e-37
    assert (err <= bound).all(), f"{what}: {np.max(err / bound)} of the bound"


# (rows, K, columns): one row and column tile of each K-split kernel and their
# neighbours, partial items (K % 256 = 64, 128, 192), one unit; then outputs
# enough for the 256 x 128 tiles, of Q4_0 and Q4_K (whole items and a partial one)
# and of Q8_0 too (whole items, and every partial one); 64 x 16 and 64 x 32 tiles
# (tests/test_kernel_choice.py)
SHAPES = [(1, 64, 17), (31, 256, 17), (33, 320, 33), (64, 512, 16), (65, 704, 65), (255, 192, 31), (1000, 128, 40),
          (2049, 768, 1601), (2300, 320, 1500), (2300, 512, 1901), (2301, 576, 1900), (2299, 384, 1901), (2300, 448, 1902),
          (8000, 256, 17), (8001, 448, 17), (8100, 512, 60), (8095, 320, 63)]


@pytest.mark.parametrize("qtype", QTYPES, ids=lambda q: QN[q])
@pytest.mark.parametrize("M,K,B", SHAPES, ids=[f"{m}x{k}-b{b}" for m, k, b in SHAPES])
@pytest.mark.parametrize("exact_x", [False, True], ids=["two-terms", "three-terms"])
def test_many_columns(qgemv, qtype, M, K, B, exact_x):
    """x stored [B, K] and, the same bits, [K, B]."""
    if K % O.QTYPE_INFO[qtype][0]:
        pytest.skip("K not a multiple of the block size")
    note(f"gemm_q {QN[qtype]} {M}x{K} B={B} exact_x={exact_x}")
    w = S.quant_weights(qtype, M, K, seed=M + K, device=DEV)
    qw = vx.QWeight(w, qtype, M, K)
    x = S.activations(B, K, seed=B, device=DEV)
    x[:, :32] = 0.0
    x[0] *= 2.0 ** -60
    x[-1] *= 2.0 ** 60
    wsp = None if exact_x else vx.QuantGemv.workspace(qw, B)
    y = torch.full((B, M), float("nan"), device=DEV)
    y2 = torch.full((M, B), float("nan"), device=DEV)
    qgemv.dispatch(y.t(), qw, x.t(), x_f32=exact_x, workspace=wsp)
    qgemv.dispatch(y2, qw, x.t().contiguous(), x_f32=exact_x, workspace=wsp)
    torch.cuda.synchronize()
    ref, mag = _reference(qtype, w, M, K, x)
    _check(y, ref, mag, K, exact_x, f"{QN[qtype]} {M}x{K} b{B}")
    assert torch.equal(y.view(torch.int32), y2.t().contiguous().view(torch.int32)), "the two storages of x differ"


@pytest.mark.parametrize("qtype", QTYPES, ids=lambda q: QN[q])
@pytest.mark.parametrize("M,B", [(70, 9), (2100, 1600), (2300, 1901)], ids=["k-split", "tiles", "tiles-q8_0"])
def test_non_finite_x_exact(qgemv, qtype, M, B):
    """With x kept in f32 an infinity or a NaN gives what the f32 products
    give (infinities keep their sign), in its own column only; the largest
    finite floats are not taken for infinities."""
    K = 512
    note(f"gemm_q non-finite {QN[qtype]} {M} B={B}")
    w = S.quant_weights(qtype, M, K, seed=9, device=DEV)
    x = S.activations(B, K, seed=10, device=DEV)
    x[0, 77] = float("inf")
    x[1, 500] = -float("inf")
    x[2, 3] = float("nan")
    x[3, 128] = torch.finfo(torch.float32).max
    y = torch.empty((B, M), device=DEV)
    qgemv.dispatch(y.t(), vx.QWeight(w, qtype, M, K), x.t(), x_f32=True)
    torch.cuda.synchronize()
    wd = O.dequant(qtype, w.cpu().numpy(), M, K).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = np.array([(x[b].cpu().numpy().astype(np.float64) * wd).sum(-1) for b in range(4)])
        ref32 = ref.astype(np.float32)
    got = y[:4].cpu().numpy()
    near = np.abs(ref[3]) > 3.3e38  # rows whose result is at the edge of f32
    assert np.array_equal(np.isnan(got[:3]), np.isnan(ref32[:3]))
    assert np.array_equal(got[:2][np.isinf(ref32[:2])], ref32[:2][np.isinf(ref32[:2])])
    assert np.allclose(got[3][~near], ref[3][~near], rtol=1e-4, atol=1e33)
    assert torch.isfinite(y[4:]).all()


@pytest.mark.parametrize("qtype", QTYPES, ids=lambda q: QN[q])
def test_non_finite_x_two_terms(qgemv, qtype):
    """With a workspace a non-finite x makes its whole column non-finite and
    leaves the others as they are, as the int8 split does."""
    M, K, B = 130, 512, 40
    note(f"gemm_q non-finite two terms {QN[qtype]}")
    w = vx.QWeight(S.quant_weights(qtype, M, K, seed=9, device=DEV), qtype, M, K)
    x = S.activations(B, K, seed=10, device=DEV)
    wsp = vx.QuantGemv.workspace(w, B)
    y0, y1 = torch.empty((B, M), device=DEV), torch.empty((B, M), device=DEV)
    qgemv.dispatch(y0.t(), w, x.t(), workspace=wsp)
    x[7, 100], x[39, 511] = float("nan"), -float("inf")
    qgemv.dispatch(y1.t(), w, x.t(), workspace=wsp)
    torch.cuda.synchronize()
    good = [b for b in range(B) if b not in (7, 39)]
    assert not torch.isfinite(y1[[7, 39]]).any()
    assert torch.equal(y1[good].view(torch.int32), y0[good].view(torch.int32))


def test_padded_rows_of_w_and_y(qgemv):
    """Row stride larger than a row, y with gaps: nothing else is written."""
    M, K, B, qtype = 77, 576, 20, vx.VX_Q8_0
    note("gemm_q padded")
    w = S.quant_weights(qtype, M, K, seed=3, device=DEV)
    wp = torch.zeros((M, w.shape[1] + 20), dtype=torch.uint8, device=DEV)
    wp[:, :w.shape[1]] = w
    x = S.activations(B, K, seed=4, device=DEV)
    y = torch.full((B, 2 * M), float("nan"), device=DEV)
    qgemv.dispatch(y[:, ::2].t(), vx.QWeight(wp, qtype, M, K, row_stride=wp.shape[1]), x.t(), x_f32=True)
    torch.cuda.synchronize()
    ref, mag = _reference(qtype, w, M, K, x)
    _check(y[:, ::2], ref, mag, K, True, "padded")
    assert torch.isnan(y[:, 1::2]).all()
