"""Dequantize to rows (stride 1 along K): bit-exact against the oracle at the
edges of a workgroup's 128 groups, for any alignment of W and of the rows."""
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


@pytest.mark.parametrize("qtype", QTYPES, ids=lambda q: QN[q])
# one group, one workgroup exactly, one group more, rows shorter and longer
# than a workgroup's span
@pytest.mark.parametrize("M,K", [(1, 32), (127, 32), (16, 256), (129, 32), (3, 1376), (5, 4096), (37, 768), (2, 8192)])
@pytest.mark.parametrize("off,wpad,ypad", [(0, 0, 0), (1, 0, 1), (2, 3, 3), (7, 1, 4)])
def test_dequantize_rows(qgemv, qtype, M, K, off, wpad, ypad):
    if K % O.QTYPE_INFO[qtype][0]:
        pytest.skip("K not a multiple of the block size")
    note(f"dequantize rows {QN[qtype]} {M}x{K} off={off} pads={wpad},{ypad}")
    w = S.quant_weights(qtype, M, K, seed=M + K, device=DEV)
    nb = w.shape[1] + wpad
    buf = torch.zeros(off + M * nb, dtype=torch.uint8, device=DEV)
    buf[off:].view(M, nb)[:, :w.shape[1]] = w
    y = torch.full((M, K + ypad), float("nan"), device=DEV)
    qgemv.dequantize(y[:, :K], vx.QWeight(buf[off:], qtype, M, K, row_stride=nb))
    torch.cuda.synchronize()
    ref = O.dequant(qtype, w.cpu().numpy(), M, K)
    assert np.array_equal(y[:, :K].cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert torch.isnan(y[:, K:]).all()
