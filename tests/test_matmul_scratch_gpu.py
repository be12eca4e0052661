"""bchip_matmul where its scratch cannot be had: a fresh context's call under graph capture, where
nothing can be allocated, takes the form that needs none and gives the same bits as the eager
call with scratch, on every replay."""
import ctypes

import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu


def hip(name, *args):
    e = getattr(ctypes.CDLL("libamdhip64.so"), name)(*args)
    assert e == 0, f"{name}: {e}"


def captured(ctx, call):
    """call() captured from ctx's stream, as a launchable graph."""
    s, graph, ex = ctypes.c_void_p(ctx.stream()), ctypes.c_void_p(), ctypes.c_void_p()
    hip("hipStreamBeginCapture", s, 0)
    try:
        call()
    finally:
        e = ctypes.CDLL("libamdhip64.so").hipStreamEndCapture(s, ctypes.byref(graph))
    assert e == 0, f"hipStreamEndCapture: {e}"
    hip("hipGraphInstantiate", ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0))
    hip("hipGraphDestroy", graph)
    return s, ex


# Batches whose K splits would run in parallel (8 and 16 inputs a workgroup), and batches of the
# tile kernel with 32, 64 and 128 inputs a workgroup.
@pytest.mark.parametrize("ty", [O.F16, O.Q8_0, O.Q4K, O.Q6K], ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,n", [(1000, 4096, 3), (4100, 4096, 12), (13500, 4096, 17), (301, 2048, 2000),
                                         (8300, 2304, 65), (33000, 512, 200)])
def test_a_captured_call_without_scratch(ty, rows, cols, n):
    run(ty, rows, cols, n)


# Cols off a multiple of 256, on both sides of the 56 units whose sums k_matmul_units holds at
# once, with one K split, a few and many.
@pytest.mark.parametrize("ty", [O.F16, O.Q8_0, O.Q4_0, O.Q4_1, O.Q5_0, O.Q5_1], ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,n", [(4864, 896, 70), (333, 14304, 60), (333, 14368, 40), (65, 29568, 9),
                                         (20000, 14368, 2), (17, 43040, 33)])
def test_a_captured_call_off_a_multiple_of_256(ty, rows, cols, n):
    run(ty, rows, cols, n)


def run(ty, rows, cols, n):
    some = min(rows, 131)
    data = np.resize(np.asarray(O.random_tensor(ty, some, cols, rows + n), np.uint8).reshape(some, -1),
                     (rows, O.row_bytes(ty, cols))).reshape(-1)
    x = np.random.default_rng(cols + n).standard_normal((n, cols)).astype(np.float32)
    with bchip.Ctx(0) as eager, bchip.Ctx(0) as ctx:
        def product(c):
            bufs = c.upload(data), c.upload(x), c.zeros(n * rows * 4)
            return bufs, lambda: c.matmul(bufs[0], ty, bufs[1], bufs[2], rows, cols, n)
        mine, call = product(eager)
        call()
        want = eager.read(mine[2], (n, rows))
        assert np.isfinite(want).all() and want.any()
        bufs, call = product(ctx)
        junk = ctx.upload(np.full(n * rows, -3.0, np.float32))
        s, ex = captured(ctx, call)
        for _ in range(3):
            ctx.copy(junk, bchip.F32, bufs[2], bchip.F32, 0, n * rows)
            hip("hipGraphLaunch", ex, s)
            np.testing.assert_array_equal(ctx.read(bufs[2], (n, rows)), want)
        call()  # eager, with scratch
        np.testing.assert_array_equal(ctx.read(bufs[2], (n, rows)), want)
        hip("hipGraphExecDestroy", ex)
