"""The device sampler's serial f32 sums (run_chunk in sample.hip), at the sizes where its
workgroup scan, the histogram's bound, the sort in LDS and the sort through memory begin and
end, against the CPU restatement. top_p set to a row's own running mass at some token, and to
the next f32 above it, moves the nucleus by a token if any of the steps before rounds
differently; the draws over many steps then reach its last tokens."""
import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = bchip.Ctx(0)
    yield c
    c.close()


def ids_of(ctx, scores, temperature, top_p, seed, step0):
    rows, vocab = scores.shape
    sb, ib = ctx.upload(np.ascontiguousarray(scores, np.float32)), ctx.zeros(rows * 4)
    ctx.sample(sb, rows, vocab, temperature, top_p, seed, step0, ib)
    ids = ctx.read(ib, (rows,), np.uint32)
    sb.free()
    ib.free()
    return ids


def masses(scores, temperature):
    """The running masses of one row as sample.rs sums them (f32, serial)."""
    p = np.exp(((scores - scores.max()) / np.float32(temperature)).astype(np.float64)).astype(np.float32)
    total = np.float32(0)
    for x in p:
        total += x
    q = np.sort(p)[::-1] / total
    return np.add.accumulate(q, dtype=np.float32)


@pytest.mark.parametrize("vocab", [1, 2, 511, 513, 1023, 1024, 4096, 4097, 8192, 8193, 16385, 40000])
@pytest.mark.parametrize("spread", [0.3, 2.0])
def test_the_nucleus_ends_at_the_token(ctx, vocab, spread):
    rng = np.random.default_rng(vocab)
    row = (rng.standard_normal(vocab) * spread).astype(np.float32)
    mass = masses(row, 0.8)
    scores = np.repeat(row[None], 24, axis=0)
    # (511 and 512: the last candidate whose sums one lane takes, and the first beyond)
    for k in {0, min(5, vocab - 1), min(511, vocab - 1), min(512, vocab - 1), vocab // 3, vocab // 2}:
        for top_p in (mass[k], np.nextafter(mass[k], np.float32(2))):
            got = ids_of(ctx, scores, 0.8, float(top_p), 99, 7)
            want = [O.sample(row, 0.8, float(top_p), 99, 7 + r) for r in range(24)]
            np.testing.assert_array_equal(got, np.array(want, np.uint32), err_msg=f"k {k} top_p {top_p}")


@pytest.mark.parametrize("vocab", [300, 5000, 20000])
def test_rows_with_nans_infinities_and_zeros(ctx, vocab):
    rng = np.random.default_rng(3)
    s = (rng.standard_normal((5, vocab)) * 2).astype(np.float32)
    s[0, [7, vocab - 3]] = np.nan          # NaN scores: the first of them
    s[1, :] = -1000.0
    s[1, vocab // 2] = 50.0                # one token with all the mass, the rest 0
    s[2, : vocab // 2] = -np.inf           # half the vocabulary ruled out
    s[3, :] = 1.25                         # every p is 1
    s[4] = np.sort(s[4])                   # ascending: total crosses every binade in turn
    for top_p in (0.3, 0.9, 1.0):
        got = ids_of(ctx, s, 1.0, top_p, 5, 40)
        want = [O.sample(s[r], 1.0, top_p, 5, 40 + r) for r in range(5)]
        np.testing.assert_array_equal(got, np.array(want, np.uint32), err_msg=f"top_p {top_p}")


@pytest.mark.parametrize("vocab", [300, 8192, 8193, 40000])
def test_top_p_at_or_below_zero_keeps_the_first_token(ctx, vocab):
    """A running mass of nothing already reaches such a top_p, but at least one token is kept. The
    scratch holds another call's keys, whose ids are not the answer. (NaN: no mass reaches it.)"""
    rng = np.random.default_rng(vocab)
    s = (rng.standard_normal((4, vocab)) * 2).astype(np.float32)
    s[3] = -5.0
    s[3, [vocab // 3, vocab - 1]] = 40.0  # two tokens of p = 1, all others next to 0
    ids_of(ctx, s[:, ::-1] * np.float32(0.5), 0.7, 1.0, 1, 0)
    for top_p in (0.0, -0.0, -1.0, -np.inf, np.nan, 2.0):
        got = ids_of(ctx, s, 0.9, top_p, 11, 3)
        want = [O.sample(s[r], 0.9, top_p, 11, 3 + r) for r in range(4)]
        np.testing.assert_array_equal(got, np.array(want, np.uint32), err_msg=f"top_p {top_p}")
        if top_p <= 0:
            np.testing.assert_array_equal(got, s.argmax(axis=1))
