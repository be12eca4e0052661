"""bchip_matmul's one-row kernel of the block formats (k_matmul_row) against the f64 product.
Sizes sit at its edges: weight rows off a multiple of 16 on both sides of the eight and sixteen
waves' limit, one unit, fewer units than waves, several a wave with a remainder, the most units it
takes and one more (the vector-unit pass)."""
import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu

TYPES = [O.Q8_0, O.Q4_0, O.Q4_1, O.Q5_0, O.Q5_1, O.Q4K, O.Q5K, O.Q6K]


@pytest.fixture(scope="module")
def ctx():
    c = bchip.Ctx(0)
    yield c
    c.close()


@pytest.mark.parametrize("ty", TYPES, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 1024), (33, 4096), (130, 5888), (47, 6144), (257, 14336),
                                       (4095, 4352), (4096, 4096), (4097, 1792), (4111, 4352), (17, 65536), (17, 65792)])
def test_one_row(ctx, ty, rows, cols):
    # (a block of random rows repeated: random_tensor draws slowly)
    some = min(rows, 67 if cols < 60000 else 5)
    data = np.resize(np.asarray(O.random_tensor(ty, some, cols, rows + cols), np.uint8).reshape(some, -1),
                     (rows, O.row_bytes(ty, cols))).reshape(-1)
    x = np.random.default_rng(rows).standard_normal((2, cols)).astype(np.float32)
    x[1, :cols // 2] *= 1e-5
    wb, got = ctx.upload(data), []
    for part in (x[:1], x[1:], x[:1], x[1:]):
        n = len(part)
        xb, ob = ctx.upload(np.ascontiguousarray(part)), ctx.zeros((n * rows + 64) * 4)
        ctx.matmul(wb, ty, xb, ob, rows, cols, n)
        out = ctx.read(ob, (n * rows + 64,))
        assert not out[n * rows:].any()  # nothing past the last row
        got.append(out[:n * rows].reshape(n, rows))
        xb.free()
        ob.free()
    wb.free()
    one, again = np.concatenate(got[:2]), np.concatenate(got[2:])
    np.testing.assert_array_equal(one, again)
    # x in two f16 parts (2^-22 of a term), f32 sums of a unit's 256 products in some order and a
    # few roundings after them, 64 bits from there (cols 2^-24 where the vector-unit pass takes it). |a q|
    # and |b| of a SUM format's weight can each exceed |a q + b|, at most 31-fold.
    w = O.dequant(ty, data.reshape(rows, -1)[:some].reshape(-1), some, cols).astype(np.float64)
    want = np.resize((x.astype(np.float64) @ w.T).T, (rows, 2)).T
    sizes = (np.abs(x.astype(np.float64)) @ np.abs(w).T).max(axis=1, keepdims=True)
    if ty in (O.Q4_1, O.Q5_1, O.Q4K, O.Q5K):
        sizes = sizes * 32
    chain = 264 if cols // 256 <= 256 else cols / 16 + 40
    assert (np.abs(one - want) <= (2.0 ** -22 + chain * 2.0 ** -24) * sizes).all()
