"""Quantized products with many columns: every output is written once and
right for any number of tiles of rows and columns (their order over the XCDs)."""
import pytest
import torch

import vortx_amd as vx

pytestmark = pytest.mark.gpu
BLOCK = {vx.VX_Q4_0: (32, 18), vx.VX_Q8_0: (32, 34), vx.VX_Q4_K: (256, 144)}


@pytest.mark.parametrize("qtype", list(BLOCK), ids=["q4_0", "q8_0", "q4_k"])
@pytest.mark.parametrize("M,B", [(1, 17), (33, 300), (339, 318), (65, 129), (2300, 33), (700, 7), (130, 1000), (9000, 130)])
def test_tile_counts(qgemv, qtype, M, B):
    K = 768
    qk, bb = BLOCK[qtype]
    g = torch.Generator(device="cuda").manual_seed(M + B)
    w = vx.QWeight(torch.empty(M * (K // qk) * bb, dtype=torch.uint8, device="cuda"), qtype, M, K)
    qgemv.quantize(w, torch.randn(M, K, device="cuda", generator=g))
    x = torch.randn(B, K, device="cuda", generator=g)
    wd = torch.empty(M, K, device="cuda")
    qgemv.dequantize(wd, w)
    want = x.double() @ wd.double().t()
    # f32 sums of exact products (a few roundings per block and addition), plus
    # Q4_K's offsets, up to twice the row's largest weight
    scale = wd.abs().double() if qtype != vx.VX_Q4_K else wd.abs().amax(1, keepdim=True).double().expand(M, K) * 2
    bound = (K // 8) * 2.0 ** -24 * (x.abs().double() @ scale.t())
    y = torch.full((B, M), float("nan"), device="cuda")
    qgemv.dispatch(y.t(), w, x.t(), x_f32=True)
    assert ((y.double() - want).abs() <= bound).all()
    y.fill_(float("nan"))
    qgemv.dispatch(y.t(), w, x.t(), workspace=vx.QuantGemv.workspace(w, B))
    # x rounded: to 1.6e-5 of its block's largest at worst
    amp = x.view(B, K // 32, 32).abs().amax(-1, keepdim=True).expand(B, K // 32, 32).reshape(B, K)
    assert ((y.double() - want).abs() <= bound + 1.6e-5 * (amp.double() @ wd.abs().double().t())).all()
