"""What the product that makes its rows from a 32-bit stream refuses before it looks for a GPU: results that lie on what other workgroups read."""

import ctypes

import pytest
import torch

from llmserve.ops import library

N, K = 8, 64
BYTES = 4 * N * K


def operands():
    """x, y, x_out, h_out, out and a spare, one behind the other in one buffer of float32 rows."""
    pool = torch.zeros(8, N, K)
    return pool, pool[0], pool[1], pool[2], pool[3].view(-1).view(torch.bfloat16)[: N * K].view(N, K), pool[4]


def call(x, y, x_out, h_out, out):
    weight, w = torch.ones(K), torch.zeros(K, K, dtype=torch.bfloat16)
    library.gemm_decode_stream(out, x, w, joins=(y, weight, 1e-5, x_out), h_out=h_out)


def shifted(pool, start, dtype=torch.float32):
    """[N, K] from `start` bytes of the buffer on."""
    return pool.view(-1).view(dtype)[start // torch.empty(0, dtype=dtype).element_size():][: N * K].view(N, K)


@pytest.mark.parametrize("what,place", [("x_out", 0), ("x_out", BYTES), ("x_out", 16), ("x_out", BYTES - 16), ("x_out", 2 * BYTES - 16),
                                        ("h_out", 0), ("h_out", BYTES + 16), ("h_out", 3 * BYTES - 16), ("out", 0), ("out", BYTES), ("out", 2 * BYTES),
                                        ("out", 4 * BYTES - 2 * BYTES // 4 - 16)])
def test_results_on_operands_are_refused(what, place):
    """The first of x, of y, a few numbers further on, their last ones, and other results."""
    pool, x, y, x_out, h_out, out = operands()
    moved = shifted(pool, place, torch.bfloat16 if what == "h_out" else torch.float32)
    given = dict(x=x, y=y, x_out=x_out, h_out=h_out, out=out, **{}) | {what: moved}
    with pytest.raises(ValueError, match="overlaps"):
        call(**given)


def test_results_beside_operands_are_not():
    """(the next check is for the GPU: nothing here is on one)"""
    _, x, y, x_out, h_out, out = operands()
    with pytest.raises(ValueError, match="GPU tensors only"):
        call(x, y, x_out, h_out, out)


def test_rows_of_the_result_may_have_other_things_between_them():
    both = torch.zeros(3 * N, 2 * K)
    _, x, y, x_out, h_out, _ = operands()
    with pytest.raises(ValueError, match="GPU tensors only"):
        call(x, y, x_out, h_out, both[:N, K:])


def needs_no_gpu():
    if torch.cuda.is_available():
        pytest.skip("the launchers' refusals, with addresses that nothing lies at")


@pytest.mark.parametrize("x_out,h_out,out,refused", [(3, 4, 5, False), (1, 4, 5, True), (2, 4, 5, True), (3, 1, 5, True), (3, 2, 5, True), (3, 3, 5, True),
                                                     (3, 4, 1, True), (3, 4, 2, True), (3, 4, 3, True), (3, 4, 4, True)])
def test_the_launcher_refuses_them_too(x_out, h_out, out, refused):
    """Status 1 is a refusal; without a GPU a launch ends in status 2."""
    needs_no_gpu()
    at = [ctypes.c_void_p(i * (1 << 20)) for i in range(9)]
    i, f = ctypes.c_int, ctypes.c_float
    status = library.load("gemm_decode").llms_gemm_decode_stream(
        i(0), i(0), at[out], i(K), at[6], None, i(N), i(K), i(K), i(0), i(0), f(0), i(1), at[1], at[x_out], at[h_out], at[2], at[7], f(0), f(1e-5),
        i(256), None)
    assert status == (1 if refused else 2)


@pytest.mark.parametrize("m,k,norm,ldr,refused", [(8, 2048, False, 64, False), (16, 5632, False, 64, False), (8, 2048, True, 64, True),
                                                  (16, 5632, True, 64, True), (16, 2048, False, 1 << 27, True)])
def test_a_32_bit_residual_takes_no_norm(m, k, norm, ldr, refused):
    needs_no_gpu()
    at = [ctypes.c_void_p(i * (1 << 24)) for i in range(9)]
    i, f = ctypes.c_int, ctypes.c_float
    status = library.load("gemm_decode").llms_gemm_decode(
        i(0), i(3), None, i(0), at[1], i(k), at[2], None, at[3] if norm else None, f(1e-5), i(m), i(64), i(k), i(0), i(0), i(0), i(0), i(0), None, None,
        None, None, None, None, at[4], i(ldr), i(256), i(1), i(0), f(0), None, i(0), i(0), None, None)
    assert status == (1 if refused else 2)
