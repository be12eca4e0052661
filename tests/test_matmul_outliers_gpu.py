"""bchip_matmul where 16 columns of every input row are 1e6 or 1e8 times the others and meet weights
of 0: what is left is the others' product, which the matrix cores' two-part inputs (one scale for
256 columns) must still hold to f32 rounding."""
import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu

BIG = 16  # columns


@pytest.fixture(scope="module")
def ctx():
    c = bchip.Ctx(0)
    yield c
    c.close()


def weights(ty, rows, cols):
    """Random weights, those of the first BIG columns 0: by their quants, or (K-quants) by the scale
    and the min of the block's first 32 columns."""
    w = np.array(O.random_tensor(ty, rows, cols, 9), np.uint8).reshape(rows, -1)
    if ty == O.F16:
        w[:, :2 * BIG] = 0
    elif ty == O.Q8_0:
        w[:, 2:2 + BIG] = 0
    elif ty == O.Q4_0:  # 8 in the low nibbles
        w[:, 2:2 + BIG] = (w[:, 2:2 + BIG] & 0xf0) | 8
    elif ty == O.Q5_0:  # 16: 0 in the low nibbles, 1 in qh's bits 0 .. 15
        w[:, 2:4] = 0xff
        w[:, 6:6 + BIG] &= 0xf0
    elif ty in (O.Q4K, O.Q5K):
        w[:, [4, 8]] &= 0xc0
    return w.reshape(-1)


# One row (k_matmul_row), 8 and 16 inputs a workgroup (k_matmul_mm), the tile kernel, and off a
# multiple of 256 (k_matmul_units, k_matmul_tile; the 32-weight formats and F16).
BLOCK32 = [O.Q8_0, O.Q4_0, O.Q5_0, O.F16]
CASES = [(ty, *shape) for shape in ((512, 4096, 1), (512, 256, 1), (512, 4096, 4), (2048, 4096, 12), (3100, 4096, 120))
         for ty in BLOCK32 + [O.Q4K, O.Q5K]]
CASES += [(ty, *shape) for shape in ((512, 896, 4), (2200, 896, 120)) for ty in BLOCK32]


@pytest.mark.parametrize("ty,rows,cols,n", CASES, ids=[f"{O.TYPE_NAMES[c[0]]}-{c[1]}-{c[2]}-{c[3]}" for c in CASES])
def test_columns_beside_much_larger_ones(ctx, ty, rows, cols, n):
    data = weights(ty, rows, cols)
    w = O.dequant(ty, data, rows, cols).astype(np.float64)
    assert not w[:, :BIG].any() and w[:, BIG:].any()
    wb, ob = ctx.upload(data), ctx.zeros(n * rows * 4)
    for factor in (1.0, 1e6, 1e8):
        x = np.random.default_rng(cols + n).standard_normal((n, cols)).astype(np.float32)
        x[:, :BIG] *= np.float32(factor)
        xb = ctx.upload(x)
        ctx.matmul(wb, ty, xb, ob, rows, cols, n)
        got, want = ctx.read(ob, (n, rows)), x.astype(np.float64) @ w.T
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"{O.TYPE_NAMES[ty]} {rows}x{cols} n {n} factor {factor:g}: {err:.2e}", flush=True)
        # A term is off by 2^-23 at most (x's 22 bits), 2^-24.8 in the mean square; a sum of f32
        # roundings at most one a group of 32, each 2^-24 of a partial sum: 2^-22 holds both. The
        # K-quants' a q and b are each about twice a q + b.
        assert err < (2.0 ** -21 if ty in (O.Q4K, O.Q5K) else 2.0 ** -22)
        xb.free()
    wb.free()
    ob.free()
