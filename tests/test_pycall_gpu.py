"""The binding's two ways into the library, csrc/vx_pycall.cpp for plain
tensors and ctypes for everything else, give the same bits and the same errors."""
import pytest
import torch

import vortx_amd as vx
from vortx_amd import _pycall

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    g, q, c = vx.Gemm(), vx.QuantGemv(), vx.Contiguous()
    yield g, q, c
    for o in (g, q, c):
        o.close()


def _pair(t):
    """The same view as (buffer, layout): always the ctypes path."""
    buf = t.as_strided((t.untyped_storage().nbytes() // 4,), (1,), 0)
    return buf, vx.TensorLayout(tuple(t.shape), tuple(t.stride()), t.dim(), t.storage_offset())


def _views():
    a = torch.randn(3, 70, 96, device="cuda")
    b = torch.randn(3, 96, 80, device="cuda")
    yield a, b
    yield a[1], b[2]                                          # offsets
    yield a.transpose(1, 2)[:, :64, :], torch.randn(3, 70, 80, device="cuda")
    yield a[:, 1::2, 3:67], b[:, 5:69, ::3]                   # steps
    yield a[:1, 0:1, :].expand(3, 33, 96), b                  # stride 0


@pytest.mark.parametrize("i", range(5))
def test_gemm_same_bits(ops, i):
    g = ops[0]
    a, b = list(_views())[i]
    shape = tuple(a.shape[:-1]) + (b.shape[-1],)
    outs = [torch.full(shape, 7.0, device="cuda") for _ in range(4)]
    g.dispatch(outs[0], a, b)
    g.dispatch(_pair(outs[1]), _pair(a), _pair(b))
    g.dispatch_ex(outs[2], a, b, alpha=0.5, beta=2)
    g.dispatch_ex(_pair(outs[3]), _pair(a), _pair(b), alpha=0.5, beta=2)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[2], outs[3])
    want = a.double() @ b.double()  # |error| <= K eps sum|a||b|
    bound = (a.shape[-1] + 4) * 2.0 ** -23 * (a.double().abs() @ b.double().abs())
    assert ((outs[0].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("B,ws", [(1, False), (3, False), (3, True), (9, True)])
def test_gemv_dequantize_quantize_same_bits(ops, B, ws):
    q = ops[1]
    rows, cols = 70, 512
    x = torch.randn(cols, rows + 1, device="cuda")[:, 1:].t()  # [rows, cols], strided, at an offset
    wa, wb = (vx.QWeight(torch.zeros(rows * cols // 32 * 18, dtype=torch.uint8, device="cuda"), vx.VX_Q4_0, rows, cols)
              for _ in range(2))
    q.quantize(wa, x)
    q.quantize(wb, _pair(x))
    assert torch.equal(wa.data, wb.data)
    da, db = torch.empty(cols, rows, device="cuda").t(), torch.empty(cols, rows, device="cuda").t()
    q.dequantize(da, wa)
    q.dequantize(_pair(db), wa)
    assert torch.equal(da, db)
    xb = torch.randn(B, cols, device="cuda").t()
    w = torch.empty(q.workspace_size(wa, B), dtype=torch.uint8, device="cuda") if ws else None
    ya, yb = torch.empty(B, rows, device="cuda").t(), torch.empty(B, rows, device="cuda").t()
    q.dispatch(ya, wa, xb, workspace=w)
    q.dispatch(_pair(yb), wa, _pair(xb), workspace=w)
    assert torch.equal(ya, yb)


@pytest.mark.parametrize("dtype", [torch.float32, torch.int32])
def test_contiguous_same_bits(ops, dtype):
    src = torch.arange(2 * 6 * 10 * 14, device="cuda").to(dtype).view(2, 6, 10, 14)[:, 1:, :, 2:].permute(0, 3, 1, 2)
    oa, ob = torch.zeros(src.shape, dtype=dtype, device="cuda"), torch.zeros(src.shape, dtype=dtype, device="cuda")
    ops[2].launch(oa, src)
    ops[2].launch(_pair(ob), _pair(src))
    assert torch.equal(oa, src) and torch.equal(ob, src)


def test_streams(ops):
    a, b = torch.randn(64, 64, device="cuda"), torch.randn(64, 64, device="cuda")
    want = torch.empty(64, 64, device="cuda")
    ops[0].dispatch(want, a, b)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    outs = [torch.zeros(64, 64, device="cuda") for _ in range(3)]
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops[0].dispatch(outs[0], a, b)               # the current stream
    ops[0].dispatch(outs[1], a, b, stream=s)
    ops[0].dispatch(outs[2], a, b, stream=s.cuda_stream)  # an integer: the ctypes path
    s.synchronize()
    assert all(torch.equal(o, want) for o in outs)
    graph = torch.cuda.CUDAGraph()
    out = torch.zeros(64, 64, device="cuda")
    with torch.cuda.graph(graph):                    # the current stream is the capturing one
        ops[0].dispatch(out, a, b)
    assert out.abs().max() == 0
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_unusual_operands_take_the_other_path(ops):
    g, q = ops[:2]
    a = torch.randn(64, 64, device="cuda")
    out = torch.empty(64, 64, device="cuda")
    call = lambda o, l, r, ctx=None: _pycall.gemm(vx._GEMM, ctx or g._ctx, None, o, l, r)
    assert call(out, a, a) == 0
    for bad in (a.double(), a.cpu(), a.to(torch.int32), torch.nn.Parameter(a), _pair(a), None, a.expand(1, 1, 1, 64, 64),
                a[:, :0]):
        assert call(out, a, bad) is None
    want = out.clone()
    g.dispatch(out.zero_(), a, torch.nn.Parameter(a))  # a subclass: as before
    assert torch.equal(out, want)
    for bad, err in ((a.double(), TypeError), (a.cpu(), TypeError), (a.to(torch.int32), TypeError), (None, TypeError),
                     (a.expand(1, 1, 1, 64, 64), vx.VortxError), (a[:, :3], vx.VortxError), (a[:9], vx.VortxError)):
        with pytest.raises(err):
            g.dispatch(out, bad, a)
    with pytest.raises(vx.VortxError):  # K = 0 against K = 64
        g.dispatch(out, a[:, :0], a)
    w = vx.QWeight(torch.zeros(8 * 144, dtype=torch.uint8, device="cuda"), vx.VX_Q4_0, 8, 256)
    x, y = torch.randn(256, 2, device="cuda"), torch.empty(8, 2, device="cuda")
    for ws in (torch.empty(64, dtype=torch.uint8), torch.empty(64, 64, device="cuda").t(), 3):
        with pytest.raises(TypeError):
            q.dispatch(y, w, x, workspace=ws)
    closed = vx.Gemm()
    closed.close()
    with pytest.raises(vx.VortxError):
        closed.dispatch(out, a, a)
