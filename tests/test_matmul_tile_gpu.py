"""bchip_matmul's kernels for large batches (k_matmul_tile) and for 32-weight formats whose
cols is no multiple of 256 (k_matmul_units, k_matmul_tile) against the small batches of
k_matmul_mm and each other: the same bits, since all run an output's operations in one order. Sizes sit at the
edges of its tiles: 32 and 64 input rows, 128 weight rows, steps of 64 columns (odd groups
too), K splits run in parallel and in turn, one unit and several a split."""
import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu

BLOCK32 = [O.F16, O.Q8_0, O.Q4_0, O.Q4_1, O.Q5_0, O.Q5_1]
TILE_TYPES = BLOCK32 + [O.Q4K, O.Q5K, O.Q6K]


@pytest.fixture(scope="module")
def ctx():
    c = bchip.Ctx(0)
    yield c
    c.close()


def product(ctx, ty, data, rows, cols, x):
    return products(ctx, ty, data, rows, cols, [x])[0]


def products(ctx, ty, data, rows, cols, batches):
    """The product of each batch of input rows, the weights uploaded once."""
    wb, got = ctx.upload(data), []
    for x in batches:
        xb, ob = ctx.upload(np.ascontiguousarray(x, np.float32)), ctx.zeros(len(x) * rows * 4)
        ctx.matmul(wb, ty, xb, ob, rows, cols, len(x))
        got.append(ctx.read(ob, (len(x), rows)))
        xb.free()
        ob.free()
    wb.free()
    return got


# rows x cols x n above the tile kernel's thresholds (0.1 to 1.2 G by format; the first five reach it
# for some, the others for all): 32 and 64 and 128 input rows a workgroup; K splits in parallel (up to
# 128 tiles, 255 of 32 input rows) and in turn; one unit, a few, remainders of every size.
@pytest.mark.parametrize("ty", TILE_TYPES, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,n", [(11650, 4096, 17), (5801, 4096, 32), (301, 1280, 2000), (8300, 1536, 65),
                                         (33000, 256, 100), (32900, 768, 129), (9200, 4096, 32), (301, 2048, 2000),
                                         (8300, 2304, 120), (47000, 256, 100), (32900, 768, 220), (16600, 2560, 31),
                                         (33000, 1280, 32)])
def test_tile_gives_the_small_batches_bits(ctx, ty, rows, cols, n):
    # (a block of random rows repeated: random_tensor draws slowly)
    some = 257
    data = np.resize(np.asarray(O.random_tensor(ty, some, cols, rows + n), np.uint8).reshape(some, -1),
                     (rows, O.row_bytes(ty, cols))).reshape(-1)
    x = np.random.default_rng(cols + n).standard_normal((n, cols)).astype(np.float32)
    at = [0, 15, n - 16] + ([n // 2] if n > 64 else [])  # batches of 16, 2 and 9 rows at the ends and inside
    cuts = [(k, k + size) for k, size in zip(at, (16, 2, 16, 9))]
    whole, *parts = products(ctx, ty, data, rows, cols, [x] + [x[a:b] for a, b in cuts])
    assert np.isfinite(whole).all()
    for (a, b), part in zip(cuts, parts):
        np.testing.assert_array_equal(part, whole[a:b], err_msg=f"rows {a}..{b}")


@pytest.mark.parametrize("ty", BLOCK32, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols", [(3, 32), (130, 96), (65, 896), (128, 864), (31, 2080), (17, 4384)])
def test_cols_off_a_multiple_of_256(ctx, ty, rows, cols):
    """k_matmul_units: a row's bits do not depend on its batch, and its error against the f64 product stays below what its roundings can add
    up to: x in two f16 parts (2^-22 of a term), f32 sums of a group's 32 products in some
    order (32 x 2^-24 of their sizes), two roundings a group and unit after that."""
    n = 70
    data = O.random_tensor(ty, rows, cols, 5 * rows + n)
    x = np.random.default_rng(cols).standard_normal((n, cols)).astype(np.float32)
    x[1] *= 1e-6
    x[2] *= 3e7
    whole = product(ctx, ty, data, rows, cols, x)
    for lo, hi in ((0, 2), (1, 4), (0, 8), (3, 19), (60, 70), (5, 38)):
        np.testing.assert_array_equal(product(ctx, ty, data, rows, cols, x[lo:hi]), whole[lo:hi], err_msg=f"rows {lo}..{hi}")
    w = O.dequant(ty, np.asarray(data, np.uint8).reshape(-1), rows, cols).astype(np.float64)
    sizes = np.abs(x.astype(np.float64)) @ np.abs(w).T
    # (SUM formats: |a q| and |b| of a weight can each exceed |a q + b|, at most 31-fold)
    if ty in (O.Q4_1, O.Q5_1):
        sizes = sizes.max(axis=1, keepdims=True) * 32
    bound = (2.0 ** -22 + (32 + 4 + cols / 16) * 2.0 ** -24) * sizes
    err = np.abs(whole - O.matmul_f64(ty, data, rows, cols, x, n))
    norm = np.linalg.norm(err, axis=1) / np.linalg.norm(whole, axis=1)
    print(f"{O.TYPE_NAMES[ty]} {rows}x{cols}: {norm.max():.2e}", flush=True)
    assert (err <= bound).all()
    # Of an input row's outputs together (x's high part alone is 1e-4 off, a lost or misscaled unit
    # more; three outputs may be small beside their terms).
    assert (norm < (2.0 ** -16 if rows < 64 else 2.0 ** -20)).all()


# From 0.2 G multiply-adds off a multiple of 256 the tile kernel: short last units of one and of several
# steps, odd groups, more units than a split.
@pytest.mark.parametrize("ty", BLOCK32, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,n", [(4900, 896, 70), (40000, 96, 65), (3100, 2080, 33), (700, 4832, 100)])
def test_tiles_off_a_multiple_of_256(ctx, ty, rows, cols, n):
    some = 131
    data = np.resize(np.asarray(O.random_tensor(ty, some, cols, rows + n), np.uint8).reshape(some, -1),
                     (rows, O.row_bytes(ty, cols))).reshape(-1)
    x = np.random.default_rng(cols + n).standard_normal((n, cols)).astype(np.float32)
    whole, *parts = products(ctx, ty, data, rows, cols, [x, x[:16], x[n - 9:]])
    np.testing.assert_array_equal(parts[0], whole[:16])
    np.testing.assert_array_equal(parts[1], whole[n - 9:])
    assert np.isfinite(whole).all()


# Batches of more than one slab of input rows: 256 MiB of prepared x (4608 rows of 14336 columns),
# and 262016 rows where narrow inputs would fit more.
@pytest.mark.parametrize("ty,rows,cols,n,slab", [(O.Q4K, 256, 14336, 4700, 4608), (O.Q8_0, 130, 14336, 9300, 4608),
                                                 (O.F16, 12, 256, 262500, 262016), (O.Q8_0, 17, 96, 524280, 262016)],
                         ids=str)
def test_slabs_give_the_small_batches_bits(ctx, ty, rows, cols, n, slab):
    wb = ctx.upload(np.asarray(O.random_tensor(ty, rows, cols, 3), np.uint8))
    xb, ob, part = ctx.zeros(n * cols * 4), ctx.zeros(n * rows * 4), ctx.zeros(16 * rows * 4)
    ctx.fill_normal(xb, bchip.F32, n * cols, 5)
    ctx.matmul(wb, ty, xb, ob, rows, cols, n)
    for at in (0, slab - 16, slab - 5, slab, 2 * slab - 8, n - 16):
        at = min(at, n - 16)
        got = ctx.read(ob, (16, rows), off=at * rows * 4)
        assert got.all() and np.isfinite(got).all()
        xs = ctx.upload(ctx.read(xb, (16, cols), off=at * cols * 4))
        ctx.matmul(wb, ty, xs, part, rows, cols, 16)
        np.testing.assert_array_equal(got, ctx.read(part, (16, rows)), err_msg=f"rows from {at}")
        xs.free()
    for b in (wb, xb, ob, part):
        b.free()


# k_matmul_mm with sixteen inputs a workgroup (splits of two units or more for Q6K, of three for Q8_0,
# Q5_0, Q5K and Q4K, the last from 1024 workgroups) and with eight on the other side of its rule.
@pytest.mark.parametrize("ty,rows,cols", [(O.Q6K, 16300, 2048), (O.Q6K, 16300, 1792), (O.Q8_0, 16300, 3072),
                                          (O.Q8_0, 16300, 2816), (O.Q5_0, 16300, 3072), (O.Q5K, 16300, 3072),
                                          (O.Q4K, 32700, 4096), (O.Q4K, 32600, 4096), (O.Q4_0, 16300, 3072)], ids=str)
def test_batches_of_9_to_16_give_the_bits_of_8(ctx, ty, rows, cols):
    some = 133
    data = np.resize(np.asarray(O.random_tensor(ty, some, cols, rows), np.uint8).reshape(some, -1),
                     (rows, O.row_bytes(ty, cols))).reshape(-1)
    x = np.random.default_rng(rows).standard_normal((16, cols)).astype(np.float32)
    first, last, *more = products(ctx, ty, data, rows, cols, [x[:8], x[8:], x, x[:9], x[4:15]])
    want = np.concatenate((first, last))
    assert np.isfinite(want).all()
    for got, (a, b) in zip(more, ((0, 16), (0, 9), (4, 15))):
        np.testing.assert_array_equal(got, want[a:b], err_msg=f"rows {a}..{b}")
