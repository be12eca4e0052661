"""bchip_matmul over F16 weights with infinities, NaN and numbers near f32's largest in x: every batch
size gives what IEEE products and sums of the row give, and no other input row moves."""
import numpy as np
import pytest

import bchip
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,n", [(300, 896, 1), (300, 896, 8), (2200, 896, 120), (300, 4096, 1), (300, 4096, 8),
                                         (2700, 4096, 70)])
def test_non_finite_inputs_of_f16_products(rows, cols, n):
    rng = np.random.default_rng(cols + n)
    w = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float16)
    w[w == 0] = 1.0
    w[5, cols // 2] = 0.0  # meets the infinity below: NaN
    clean = rng.standard_normal((n, cols)).astype(np.float32)
    x = clean.copy()
    bad = {0: [(cols // 2, np.inf)]} if n == 1 else {
        0: [(cols // 2, np.inf)], 1: [(3, -np.inf)], 2: [(7, np.nan)], 4: [(cols - 1, np.inf), (0, -np.inf)],
        5: [(cols // 2, np.inf), (cols // 2 + 1, 3e38)]}
    for row, at in bad.items():
        for col, v in at:
            x[row, col] = v
    if n > 1:
        x[6, ::7] = 1e37 * np.sign(x[6, ::7])  # (sums about 1e37: f32 holds them)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
    with bchip.Ctx(0) as ctx:
        wb, ob = ctx.upload(w.reshape(-1)), ctx.zeros(n * rows * 4)

        def product(v):
            ctx.matmul(wb, O.F16, ctx.upload(v), ob, rows, cols, n)
            return ctx.read(ob, (n, rows))
        got, before = product(x), product(clean)
    for row in range(n):
        if row in bad:
            np.testing.assert_array_equal(np.isnan(got[row]), np.isnan(want[row]), err_msg=f"row {row}")
            ok = ~np.isnan(want[row])
            np.testing.assert_array_equal(got[row][ok], want[row][ok], err_msg=f"row {row}")  # infinities
        elif row != 6:
            np.testing.assert_array_equal(got[row], before[row], err_msg=f"row {row}")
    if n > 1:
        np.testing.assert_allclose(got[6], want[6], rtol=0, atol=2.0 ** -20 * np.abs(want[6]).max())
