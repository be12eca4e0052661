"""The two forms of attention over f32 caches (one workgroup a tile and chunk; four tiles a
workgroup over the whole list) where the dispatch changes between them: a row's bits are
those of its own one-row call, a chain tree's those of the line, and the error against 64 bits
stays within the bound of the arithmetic."""
import math

import numpy as np
import pytest

import bchip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bchip.Ctx(0)
    yield c
    c.close()


def _attend(ctx, q, kc, vc, tree, rows, nh, nkv, hd, pos, masks=None):
    bufs = [ctx.upload(q), ctx.upload(kc), ctx.upload(vc), ctx.zeros(q.nbytes)]
    if masks is not None:
        bufs.append(ctx.upload(masks))
    ctx.attention(*bufs[:3], bchip.F32, bufs[3], bufs[4] if masks is not None else None, tree, rows, nh, nkv, hd, pos,
                  1.0 / math.sqrt(hd))
    out = ctx.read(bufs[3], (rows, nh, hd))
    for b in bufs:
        b.free()
    return out


def _check64(out, q, kc, vc, rows, nh, nkv, hd, pos):
    u, scale = 2.0 ** -24, 1.0 / math.sqrt(hd)
    for r in sorted({0, rows // 2, rows - 1}):
        n = pos + r + 1
        for h in sorted({0, nh - 1}):
            j = h // (nh // nkv)
            k = kc[:n].reshape(n, nkv, hd)[:, j].astype(np.float64)
            v = vc[:n].reshape(n, nkv, hd)[:, j].astype(np.float64)
            x = q.reshape(rows, nh, hd)[r, h].astype(np.float64)
            s = k @ x * scale
            w = np.exp(s - s.max())
            want = w @ v / w.sum()
            # A score: eight chains of hd / 8 rounded steps, three levels of sums, the scale, the
            # subtraction and the exponential; the weights' sums: 32 entries a block, 6 blocks a
            # chunk, then the chunks, a rounding each, and the hardware exp2's two.
            es = ((hd / 8 + 8) * (np.abs(k) @ np.abs(x)).max() * scale + 4 * np.abs(s).max()) * u
            bound = np.abs(v).max() * 2 * (2 * es + (32 + 2 * 6 + 4 * (n / 192 + 1) + 4) * u)
            assert np.abs(out[r, h] - want).max() <= bound


# (nh, nkv, hd, rows, pos): tiles below and at 512, lists within a block, a chunk and past both,
# the last workgroup's tiles cut, head dims below their padded size.
LINES = [(8, 8, 128, 1024, 3), (32, 8, 128, 253, 189), (32, 8, 128, 256, 189), (14, 2, 64, 515, 31), (16, 16, 40, 520, 160),
         (8, 8, 256, 1030, 65), (16, 1, 32, 513, 0), (28, 4, 80, 517, 383),
         # lists of at most 128 entries and one more (own calls: at most)
         (32, 8, 128, 120, 9), (14, 2, 64, 100, 28), (16, 8, 256, 110, 30), (8, 2, 32, 97, 31)]


@pytest.mark.parametrize("nh,nkv,hd,rows,pos", LINES)
def test_a_row_has_the_bits_of_its_own_call(ctx, nh, nkv, hd, rows, pos):
    print(f"f32 line {nh} {nkv} {hd}: {rows} rows at {pos}", flush=True)
    rng = np.random.default_rng(rows + hd)
    q = 2 * rng.standard_normal((rows, nh * hd), dtype=np.float32)
    kc, vc = rng.standard_normal((2, pos + rows, nkv * hd), dtype=np.float32)
    out = _attend(ctx, q, kc, vc, False, rows, nh, nkv, hd, pos)
    for r in sorted({0, 1, 62, rows // 2, rows - 2, rows - 1}):
        one = _attend(ctx, q[r:r + 1], kc, vc, False, 1, nh, nkv, hd, pos + r)
        np.testing.assert_array_equal(out[r].view(np.uint32), one[0].view(np.uint32), err_msg=f"row {r}")
    _check64(out, q, kc, vc, rows, nh, nkv, hd, pos)


# Chunks below pos, whose tiles hold several rows: none, one, several, pos at a chunk's end, one to
# sixteen heads a KV head, rows that don't fill a tile. The last: slots of more elements than the
# split form's offsets reach.
TREES = [(32, 8, 128, 40, 0), (14, 2, 64, 33, 64), (14, 2, 64, 33, 65), (8, 8, 128, 64, 300), (64, 8, 128, 63, 190), (16, 16, 64, 33, 500), (32, 8, 128, 33, 777), (28, 4, 64, 17, 1153),
         (16, 1, 32, 30, 400), (8, 2, 128, 3, 576), (40, 8, 256, 21, 575), (4100, 4100, 256, 5, 2)]


@pytest.mark.parametrize("nh,nkv,hd,rows,pos", TREES)
def test_a_chain_tree_has_the_bits_of_the_line(ctx, nh, nkv, hd, rows, pos):
    print(f"f32 tree {nh} {nkv} {hd}: {rows} rows at {pos}", flush=True)
    rng = np.random.default_rng(rows + hd)
    q = 2 * rng.standard_normal((rows, nh * hd), dtype=np.float32)
    kc, vc = rng.standard_normal((2, pos + rows, nkv * hd), dtype=np.float32)
    masks = bchip.masks_words(np.array([(1 << (r + 1)) - 1 for r in range(rows)], np.uint64))
    tree = _attend(ctx, q, kc, vc, True, rows, nh, nkv, hd, pos, masks)
    line = _attend(ctx, q, kc, vc, False, rows, nh, nkv, hd, pos)
    np.testing.assert_array_equal(tree.view(np.uint32), line.view(np.uint32))
    _check64(tree, q, kc, vc, rows, nh, nkv, hd, pos)
