"""Batched quantized products where K leaves some of a workgroup's 16 waves
without an item of 256 weights (one to three items a wave)."""
import pytest
import torch

import vortx_amd as vx
from vortx_amd import synthetic as S

pytestmark = pytest.mark.gpu
BLOCK = {vx.VX_Q4_0: (32, 18), vx.VX_Q8_0: (32, 34), vx.VX_Q4_K: (256, 144)}


@pytest.mark.parametrize("qtype", list(BLOCK), ids=["q4_0", "q8_0", "q4_k"])
@pytest.mark.parametrize("M,K,B", [(1, 256, 2), (300, 256, 16), (70, 1536, 4), (520, 1600, 8), (4700, 512, 3), (13000, 768, 9),
                                   (90, 3840, 16), (257, 4352, 4), (9000, 4608, 7), (33, 8448, 2), (40, 8448, 8)])
def test_waves_without_items(qgemv, qtype, M, K, B):
    qk, bb = BLOCK[qtype]
    K -= K % qk
    g = torch.Generator(device="cuda").manual_seed(M + K)
    w = vx.QWeight(torch.empty(M * (K // qk) * bb, dtype=torch.uint8, device="cuda"), qtype, M, K)
    qgemv.quantize(w, torch.randn(M, K, device="cuda", generator=g))
    x = S.activations(B, K, seed=B, device="cuda")
    ys = [torch.full((B, M), float("nan"), device="cuda") for _ in range(3)]
    qgemv.dispatch(ys[0].t(), w, x.t())
    qgemv.dispatch(ys[1].t(), w, x.t(), workspace=vx.QuantGemv.workspace(w, B))
    xq = vx.XQ.empty(K, B)
    qgemv.quantize_x(xq, x.t())
    qgemv.dispatch_xq(ys[2].t(), w, xq)
    wd = torch.empty(M, K, device="cuda")
    qgemv.dequantize(wd, w)
    want = x.double() @ wd.double().t()
    # x: 1.6e-5 of its block's maximum; f32 sums over K / 32 blocks of an
    # exact dot, each with a few roundings, in chunks over the waves
    xb = x.view(B, K // 32, 32)
    amp = xb.abs().amax(-1, keepdim=True).expand_as(xb).reshape(B, K)
    # Q4_K rounds sc (c2 T) and m S apart: up to 15 sc and m instead of the difference
    scale = wd.abs().double() if qtype != vx.VX_Q4_K else wd.abs().amax(1, keepdim=True).double().expand(M, K) * 2
    bound = 1.6e-5 * (amp.double() @ wd.abs().double().t()) + (K // 32 + 32) * 2.0 ** -24 * (x.abs().double() @ scale.t())
    for y in ys:
        assert ((y.double() - want).abs() <= bound).all()
