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
    # ordinary columns; half of them 1e-5 of the rest; those alone (their units' own scales)
    x = np.random.default_rng(rows).standard_normal((3, cols)).astype(np.float32)
    x[1:, :cols // 2] *= 1e-5
    x[2, cols // 2:] = 0.0
    wb, got = ctx.upload(data), []
    for part in (x[:1], x[1:2], x[2:], x[:1], x[1:2], x[2:]):
        n = len(part)
        xb, ob = ctx.upload(np.ascontiguousarray(part)), ctx.zeros((n * rows + 64) * 4)
        ctx.matmul(wb, ty, xb, ob, rows, cols, n)
        out = ctx.read(ob, (n * rows + 64,))
        assert not out[n * rows:].any()  # nothing past the last row
        got.append(out[:n * rows].reshape(n, rows))
        xb.free()
        ob.free()
    wb.free()
    one, again = np.concatenate(got[:3]), np.concatenate(got[3:])
    np.testing.assert_array_equal(one, again)
    # x in two f16 parts (at most 2^-23 of a term), f32 sums of a unit's 256 products, 64 bits from
    # there (the vector-unit pass: f32 chains): of the whole row of outputs, 2^-20 holds what the
    # roundings come to also where a q and b of a weight are several times a q + b (measured at most
    # 7e-7, one output of 256 columns). x's high part alone is 1e-4 off, and so is a small half that is lost or misscaled.
    w = O.dequant(ty, data.reshape(rows, -1)[:some].reshape(-1), some, cols).astype(np.float64)
    want = np.resize((x.astype(np.float64) @ w.T).T, (rows, 3)).T

    def off(got):
        d = got - want
        return np.linalg.norm(d, axis=1) / np.linalg.norm(want, axis=1), np.abs(d).max(axis=1) / np.sqrt((want ** 2).mean(axis=1))
    norm, most = off(one)
    print(f"{O.TYPE_NAMES[ty]} {rows}x{cols}: {norm.max():.2e}, {most.max():.2e}", flush=True)
    assert (norm < 2.0 ** -20).all() and (most < 2.0 ** -18).all()
    u = x.astype(np.float64).reshape(3, -1, 256)
    scale = 2.0 ** (14 - np.floor(np.log2(np.maximum(np.abs(u).max(axis=2, keepdims=True), 1e-30))))
    high = ((u * scale).astype(np.float16) / scale).reshape(3, -1)
    assert (off(np.resize((high @ w.T).T, (rows, 3)).T)[0] > 2.0 ** -16).all()
