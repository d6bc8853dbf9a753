"""The shapes of the GPU tests reach every kernel that the host chooses among
(on the MI355X's 256 CUs; host logic only)."""
import ctypes as C

import pytest

import vortx_amd as vx
from tests import test_gemm_bf_gpu as bf
from tests import test_gemm_bf_look_gpu as bf_look
from tests import test_gemm_k16_gpu as k16
from tests import test_gemm_q_gpu as q
from tests import test_gemm_q_look_gpu as q_look
from vortx_amd import _ffi

CUS = 256
W, N, S2, S, KS, K16 = range(6)


def _bf(M, N, K, batch=1, pin=0):
    return vx.lib().vx_plan_gemm_bf(CUS, C.c_uint32(M), C.c_uint32(N), C.c_uint32(K), C.c_uint32(batch), C.c_uint32(pin))


def _q(qtype, M, K, B, terms):
    return vx.lib().vx_plan_gemm_q(CUS, qtype, C.c_uint32(M), C.c_uint32(K), C.c_uint32(B), terms)


def _args(mark):
    return [tuple(a) for a in mark.args[1]]


def _params(f, names):
    return next(_args(m) for m in f.pytestmark if m.name == "parametrize" and m.args[0] == names)


def test_gemm_shapes_reach_every_kernel():
    # (the transposed forms are a parameter of the same tests)
    by = {}
    for s in bf.SHAPES:
        by.setdefault(_bf(*s), []).append(s)
    assert sorted(by) == [W, N, S2, S, KS, K16]
    assert {-(-K // 64) % 2 for _, _, K, _ in by[S2]} == {0, 1} and {K % 64 == 0 for _, _, K, _ in by[S2]} == {True, False}
    for shapes in (_args(bf.KERNELS.mark), _args(bf_look.SHAPES.mark), _params(bf_look.test_cost_of_non_finite_and_small, "M,N,K")):
        assert {_bf(*s) for s in shapes} == {W, N, S2, S, KS, K16}, shapes
    shapes = _params(k16.test_sizes_and_strides, "n,M,N,K")
    assert K16 in {_bf(M, N, K, n) for n, M, N, K in shapes}


def test_pinned_tile_shapes_are_taken():
    shapes = _params(bf.test_tile_shapes_give_the_same_bits, "M,N,K")
    pins = {_ffi.VX_GEMM_TILE_NARROW: {N}, _ffi.VX_GEMM_TILE_WIDE: {W}, _ffi.VX_GEMM_TILE_SMALL: {S, S2}}
    for pin, want in pins.items():
        assert {_bf(*s, pin=pin) for s in shapes} == want


@pytest.mark.parametrize("qtype", [vx.VX_Q4_0, vx.VX_Q8_0, vx.VX_Q4_K], ids=["q4_0", "q8_0", "q4_k"])
@pytest.mark.parametrize("terms", [2, 3])
def test_quantized_shapes_reach_every_kernel(qtype, terms):
    shapes = [s for s in q.SHAPES if qtype != vx.VX_Q4_K or s[1] % 256 == 0]
    by = {}
    for s in shapes:
        by.setdefault(_q(qtype, *s, terms), []).append(s)
    assert {0, 1, 2, 3} <= set(by), by
    if qtype != vx.VX_Q4_K:  # whole items, and a last one of 2, 4 and 6 blocks
        assert {K % 256 for _, K, _ in by[3]} == {0, 64, 128, 192}
    for f in (q_look.test_cost_of_non_finite_x, q_look.test_small_x_keeps_its_bits, q_look.test_large_x_with_a_workspace):
        assert 3 in {_q(qtype, M, 512, B, terms) for M, B in _params(f, "M,B")}
    assert 3 in {_q(qtype, M, 512, B, terms) for M, B in _params(q.test_non_finite_x_exact, "M,B")}
