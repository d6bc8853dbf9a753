"""VX_GEMV_X_INT8 keeps the int8 split of x at every number of columns."""
import ctypes as C

import pytest
import torch

import vortx_amd as vx
from tests.helpers import note
from vortx_amd import synthetic as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("qtype", [vx.VX_Q4_0, vx.VX_Q8_0, vx.VX_Q4_K], ids=["q4_0", "q8_0", "q4_k"])
@pytest.mark.parametrize("M,K,B", [(300, 512, 17), (2000, 1024, 40), (2300, 768, 500)])
def test_int8_is_the_split(qgemv, qtype, M, K, B):
    note(f"int8 split by name {qtype} {M}x{K} B={B}")
    w = vx.QWeight(S.quant_weights(qtype, M, K, seed=M, device=DEV), qtype, M, K)
    x = S.activations(B, K, seed=B, device=DEV)
    q = vx.XQ.empty(K, B)
    want, got, noalloc = (torch.full((B, M), float("nan"), device=DEV) for _ in range(3))
    qgemv.quantize_x(q, x.t())
    qgemv.dispatch_xq(want.t(), w, q)
    qgemv.dispatch(got.t(), w, x.t(), x_int8=True, workspace=vx.QuantGemv.workspace(w, B))
    yv, xv, wc = vx._view_of(noalloc.t(), True), vx._view_of(x.t(), False), w._c()
    assert vx.lib().vx_gemv_q_noalloc(qgemv._h, torch.cuda.current_stream().cuda_stream, C.byref(yv), C.byref(wc), C.byref(xv),
                                      vx._ffi.VX_GEMV_X_INT8) == 0
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    assert torch.equal(noalloc.view(torch.int32), want.view(torch.int32))
