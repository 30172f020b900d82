"""Q6_K and Q8_0 projections of 2048 columns (gemv_q68.hip): one weight row, whole and ragged tiles of sixteen, more tiles than
compute units; one activation row, a launch's sixteen and one more; a row so large and one so small that their binary16 parts
need the power of two; against a float64 product."""
import numpy as np
import pytest

import oracle_lib as O
import shv
from test_dequant_gpu import random_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["Q6_K", "Q8_0"])
@pytest.mark.parametrize("n,rows", [(1, 1), (16, 16), (17, 2), (4099, 17), (4096 + 4096 * 3 + 5, 5)])
def test_rows(ctx, name, n, rows):
    typ, k = O.GGML_TYPES[name], 2048
    rng = np.random.default_rng(n + rows)
    raw = random_tensor(name, n * k, seed=n)
    w = O.dequant(typ, raw, n * k).reshape(n, k).astype(np.float64)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[0] *= 1e7
    x[-1] *= 1e-9
    dw, dx, y = ctx.upload(raw), ctx.upload(x), ctx.alloc(rows * n * 4)
    ctx.gemv(typ, dw, dx, y, n, k, n_tok=rows)
    got, want = y.read(np.float32, rows * n).reshape(rows, n), x.astype(np.float64) @ w.T
    size = np.sqrt((x.astype(np.float64) ** 2) @ (w ** 2).T)  # what a sum of such terms amounts to
    assert (np.abs(got - want) <= 1e-5 * size).all()
    gamma = (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    ctx.gemv(typ, dw, dx, y, n, k, n_tok=rows, gamma=ctx.upload(gamma), eps=1e-30, residual=y)
    x64 = x.astype(np.float64)
    xn = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-30) * gamma
    size = np.sqrt((xn ** 2) @ (w ** 2).T) + np.abs(got)
    assert (np.abs(y.read(np.float32, rows * n).reshape(rows, n) - (xn @ w.T + got)) <= 1e-5 * size).all()


@pytest.mark.parametrize("name", ["Q6_K", "Q8_0"])
@pytest.mark.parametrize("rows", [1, 4, 9])
def test_infinities(ctx, name, rows):
    """A row with an infinity comes out as float32 sums give it: infinite with the weight's sign, NaN where infinities of both signs,
    a zero weight or a NaN meet; its neighbours are as they would be without it."""
    typ, n, k = O.GGML_TYPES[name], 67, 2048
    rng = np.random.default_rng(rows)
    raw = random_tensor(name, n * k, seed=n)
    w = O.dequant(typ, raw, n * k).reshape(n, k).astype(np.float64)
    x = (rng.standard_normal((rows, k)) * 1e5).astype(np.float32)
    plain = x.copy()
    x[0, 77] = np.inf
    if rows > 1:
        x[1, 5], x[1, 1029], x[2, 2047], x[3, 900] = -np.inf, np.inf, -np.inf, np.nan
    y = ctx.alloc(rows * n * 4)
    ctx.gemv(typ, ctx.upload(raw), ctx.upload(x), y, n, k, n_tok=rows)
    got = y.read(np.float32, rows * n).reshape(rows, n)
    with np.errstate(invalid="ignore"):
        want = np.stack([[(row * r).sum() for r in w] for row in x.astype(np.float64)])
    for t in range(rows):
        if np.isfinite(x[t]).all():
            size = np.sqrt((plain[t].astype(np.float64) ** 2) @ (w ** 2).T)
            assert (np.abs(got[t] - want[t]) <= 1e-5 * size).all()
        else:
            assert not np.isfinite(want[t]).any() and np.array_equal(got[t], want[t].astype(np.float32), equal_nan=True), t
    assert np.isinf(want[0]).any()
