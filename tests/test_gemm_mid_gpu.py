"""Projections of 9 to 16 and of 65 to 512 rows keep a block's weights in registers while tiles of 16 activation rows go by (gemm_mid.hip).
Here the ends of that range, ragged last tiles, several tiles a block and several blocks a tile range, weight rows that end
inside a tile, and two passes past it, in blocks of one and of two groups of 64 rows; each with a folded prologue, a residual updated in place or a ring to write, against a float64 product."""
import numpy as np
import pytest

import oracle_lib as O
import shv

pytestmark = pytest.mark.gpu
A = shv.api


@pytest.mark.parametrize("n,k,rows", [(48, 2048, 9), (12352, 2048, 65), (2048, 4096, 16), (2055, 4096, 80), (70, 2048, 512), (9216, 2048, 81),
                                      (2048, 4096, 255), (17, 4096, 511), (12352, 2048, 150), (512, 2048, 513), (200, 2048, 1050)])
def test_rows_of_a_pass(n, k, rows):
    rng = np.random.default_rng(n + k + rows)
    ctx = A.Context(0)
    try:
        wq = O.quantize_q4k((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
        w64 = O.dequant_q4k(wq, k).astype(np.float64)
        x = (rng.standard_normal((rows, k)) * rng.uniform(0.01, 30.0, size=(rows, 1))).astype(np.float32)
        gamma = (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
        x64 = x.astype(np.float64)
        want = (x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-6) * gamma) @ w64.T
        # the norm folded in, the residual in place
        res = rng.standard_normal((rows, n)).astype(np.float32)
        dw, dx, dg, dy = ctx.upload(wq), ctx.upload(x), ctx.upload(gamma), ctx.upload(res)
        ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_RMSNORM, gamma=dg, residual=dy)
        got = dy.read(np.float32, rows * n).reshape(rows, n)
        err = np.linalg.norm(got - (want + res), axis=1) / np.linalg.norm(want + res, axis=1)
        assert err.max() <= 1e-5, (int(err.argmax()), float(err.max()))
        # no prologue, written into a ring that wraps
        slots, pos = rows + 3, np.array([rows - 2], np.int32)
        ring = ctx.upload(np.full((slots, n), -7.0, np.float32))
        ctx.gemv_q4k(dw, dx, ring, n, k, n_tok=rows, pos=ctx.upload(pos), seq_len=rows, ring_slots=slots, ring_stride=n)
        got = ring.read(np.float32, slots * n).reshape(slots, n)
        at = (pos[0] + np.arange(rows)) % slots
        want = x64 @ w64.T
        err = np.linalg.norm(got[at] - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() <= 1e-5, (int(err.argmax()), float(err.max()))
        assert (np.delete(got, at, axis=0) == -7.0).all()
    finally:
        ctx.destroy()


@pytest.mark.parametrize("n,k,rows", [(300, 2048, 17), (2055, 4096, 33), (12352, 2048, 48), (2048, 4096, 49)])
def test_rows_of_a_short_prompt(n, k, rows):
    """17 to 48 rows take these kernels too; 49 the kernel of one 64-row group."""
    test_rows_of_a_pass(n, k, rows)


@pytest.mark.parametrize("rows,k,head_dim,n_seq", [(9, 2048, 4, 1), (12, 4096, 128, 3), (16, 2048, 8, 2), (40, 4096, 16, 1), (48, 2048, 32, 4), (65, 4096, 64, 5),
                                                   (66, 2048, 256, 1), (150, 4096, 128, 1), (12, 2048, 0, 2), (81, 4096, 0, 1)])
def test_gates_of_a_pass(rows, k, head_dim, n_seq):
    """The staging launch's gated prologues: every width of a head that a super-block holds, gates in rows of their own and in a ring
    that wraps, by a slot table in another order; sigmoid gates behind each head's query half and as plain rows (head_dim 0)."""
    n, rng = 40, np.random.default_rng(rows + k + head_dim)
    ctx = A.Context(0)
    try:
        wq = O.quantize_q4k((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
        w64 = O.dequant_q4k(wq, k).astype(np.float64)
        x, z = rng.standard_normal((rows, k)).astype(np.float32), (2 * rng.standard_normal((rows, k))).astype(np.float32)
        sig = 1 / (1 + np.exp(-z.astype(np.float64)))
        dw, dx, dy = ctx.upload(wq), ctx.upload(x), ctx.alloc(rows * n * 4)

        def check(want):
            want, got = want @ w64.T, dy.read(np.float32, rows * n).reshape(rows, n)
            err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
            assert err.max() <= 1e-5, (int(err.argmax()), float(err.max()))
            dy.zero()

        if head_dim == 0:
            ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_MUL_SIGMOID, z=ctx.upload(z))
            return check(x.astype(np.float64) * sig)
        pair = np.concatenate([rng.standard_normal((rows, k // head_dim, head_dim)).astype(np.float32), z.reshape(rows, -1, head_dim)], axis=2)
        ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_MUL_SIGMOID, z=ctx.upload(pair), head_dim=head_dim, z_stride=2 * k)
        check(x.astype(np.float64) * sig)
        if head_dim < 32:
            return
        gamma = (1 + 0.1 * rng.standard_normal(head_dim)).astype(np.float32)
        h = x.astype(np.float64).reshape(rows, -1, head_dim)
        want = (h / np.sqrt((h * h).mean(axis=2, keepdims=True) + 1e-6) * gamma).reshape(rows, k) * sig
        ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_GATED_NORM, gamma=ctx.upload(gamma), z=ctx.upload(z), head_dim=head_dim)
        check(want)
        seq_len, stride = rows // n_seq, k + 8
        slots, pos, slot = seq_len + 1, np.arange(n_seq, dtype=np.int32) + 1, np.arange(n_seq, 0, -1).astype(np.int32)
        ring = np.zeros((n_seq + 1, slots, stride), np.float32)
        for s in range(n_seq):
            for i in range(seq_len):
                ring[slot[s], (pos[s] + i) % slots, :k] = z[s * seq_len + i]
        ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_GATED_NORM, gamma=ctx.upload(gamma), z=ctx.upload(ring), head_dim=head_dim,
                     pos=ctx.upload(pos), slot=ctx.upload(slot), seq_len=seq_len, ring_slots=slots, ring_stride=stride, z_ring=1)
        check(want)
    finally:
        ctx.destroy()


@pytest.mark.parametrize("n,rows", [(65536, 5), (65537, 6), (65551, 8), (65536 + 8191, 9), (70000, 16), (65535, 5), (65536, 4)])
def test_few_rows_against_a_matrix_of_many_rounds(n, rows):
    """The walk over groups of sixteen weight rows: the least of them, a last group of one row and of fifteen, blocks with one group more
    than others, a matrix a row short of it and a pass; a norm folded in, residual rows, and a ring to write that wraps."""
    k, rng = 2048, np.random.default_rng(n + rows)
    ctx = A.Context(0)
    try:
        part = O.quantize_q4k((rng.standard_normal((4099, k)) * 0.02).astype(np.float32)).reshape(4099, -1)
        w64 = O.dequant_q4k(part, k).astype(np.float64).reshape(4099, k)
        of = np.arange(n) % 4099
        dw = ctx.upload(np.ascontiguousarray(part[of]))
        x = (rng.standard_normal((rows, k)) * rng.uniform(0.01, 30.0, size=(rows, 1))).astype(np.float32)
        gamma = (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
        x64, res = x.astype(np.float64), rng.standard_normal((rows, n)).astype(np.float32)
        want = ((x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-6) * gamma) @ w64.T)[:, of] + res
        dy = ctx.upload(np.concatenate([res.ravel(), np.full(64, -7.0, np.float32)]))
        ctx.gemv_q4k(dw, ctx.upload(x), dy, n, k, n_tok=rows, prologue=A.PRO_RMSNORM, gamma=ctx.upload(gamma), residual=dy)
        got = dy.read(np.float32, rows * n + 64)
        assert (got[rows * n:] == -7.0).all()
        got = got[:rows * n].reshape(rows, n)
        assert (np.linalg.norm(got - want, axis=1) <= 1e-5 * np.linalg.norm(want, axis=1)).all()
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
        slots, pos = rows + 1, np.array([rows - 1], np.int32)
        ring = ctx.upload(np.full((slots, n), -7.0, np.float32))
        ctx.gemv_q4k(dw, ctx.upload(x), ring, n, k, n_tok=rows, pos=ctx.upload(pos), seq_len=rows, ring_slots=slots, ring_stride=n)
        got, at, want = ring.read(np.float32, slots * n).reshape(slots, n), (pos[0] + np.arange(rows)) % slots, (x64 @ w64.T)[:, of]
        assert (np.linalg.norm(got[at] - want, axis=1) <= 1e-5 * np.linalg.norm(want, axis=1)).all()
        assert (np.delete(got, at, axis=0) == -7.0).all()
    finally:
        ctx.destroy()


@pytest.mark.parametrize("rows,H,E", [(128, 256, 7), (129, 1024, 31), (145, 2304, 64), (2001, 512, 32)])
def test_router_logits_of_a_long_pass(rows, H, E):
    """Columns of one super-block, of fewer than the block's waves and of more; router rows (the experts and the shared
    expert's gate) around a block's 32; whole and ragged tiles, one and several a block."""
    rng = np.random.default_rng(rows + H + E)
    ctx = A.Context(0)
    try:
        h = (rng.standard_normal((rows, H)) * 2).astype(np.float32)
        gamma = (1 + 0.1 * rng.standard_normal(H)).astype(np.float32)
        router, gate = (rng.standard_normal((E, H)) * 0.08).astype(np.float32), (rng.standard_normal(H) * 0.08).astype(np.float32)
        xn, logits = ctx.alloc(rows * H * 4), ctx.alloc(rows * (E + 1) * 4)
        args = A.MoeRouterArgs(ctx.upload(h).ptr, ctx.upload(gamma).ptr, ctx.upload(router).ptr, ctx.upload(gate).ptr, xn.ptr, logits.ptr,
                               ctx.alloc(rows * 4 * 4).ptr, ctx.alloc(rows * 5 * 4).ptr, rows, H, E, 4, 1e-6, H, 0)
        ctx.dispatch_multi([A.make_op(A.OP_MOE_ROUTER, args)])
        h64 = h.astype(np.float64)
        want = (h64 / np.sqrt((h64 * h64).mean(axis=1, keepdims=True) + 1e-6) * gamma) @ np.vstack([router, gate]).astype(np.float64).T
        got = logits.read(np.float32, rows * (E + 1)).reshape(rows, E + 1)
        assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max() * 4
    finally:
        ctx.destroy()


@pytest.mark.parametrize("rows,E,gate", [(17, 512, True), (48, 512, True), (49, 512, True), (65, 512, True), (80, 512, False), (121, 512, True), (128, 512, True), (129, 512, True), (256, 512, True), (257, 512, True),
                                         (384, 512, True), (385, 512, True), (70, 7, True), (100, 17, True), (300, 31, False), (2000, 33, True)])
def test_router_of_a_lower_pass(rows, E, gate):
    """Blocks of 16 experts, of 32, of 16 again and the staged form behind them; experts that end inside a block, fewer of them
    than a tile's tokens and columns need blocks; with and without the shared expert's gate; a row of another size beside every
    other; an infinity that stays in its row.  Sums of 2048 float32 products in chains of 16 and some ten levels over them: at
    most 26 roundings a logit of its largest partial sum, which the products' root sum of squares bounds five times over.
    All logits together: n products of size s in a chain have partial sums of s sqrt(1), s sqrt(2) .. s sqrt(n), each rounded by
    u / sqrt(3) of itself at most in the mean square (u = 2^-24).  128 chains of 16 are 17408 s^2 of u^2 / 3, the levels over them
    (four chains, four steps, eight waves) 4096, 4608 and 6144, the products h gamma, the factor and its own error 2048 s^2 a
    rounding, 5 of them: 42496 s^2 u^2 / 3 of 2048 s^2, 2.63 u.  The float32 forms give 1.9 to 2.0 u,
    the row kernel 2.2, the two halves of the staged form 3.15."""
    H, rng = 2048, np.random.default_rng(rows + E)
    ctx = A.Context(0)
    try:
        h = (rng.standard_normal((rows, H)) * rng.uniform(0.01, 30.0, size=(rows, 1))).astype(np.float32)
        bad = rows - 2
        h[bad, 77] = np.inf
        gamma = (1 + 0.1 * rng.standard_normal(H)).astype(np.float32)
        router, shared = (rng.standard_normal((E, H)) * 0.08).astype(np.float32), (rng.standard_normal(H) * 0.08).astype(np.float32)
        xn, logits = ctx.alloc(rows * H * 4), ctx.upload(np.full((rows, E + 1), -7.0, np.float32))
        args = A.MoeRouterArgs(ctx.upload(h).ptr, ctx.upload(gamma).ptr, ctx.upload(router).ptr, ctx.upload(shared).ptr if gate else None, xn.ptr, logits.ptr,
                               ctx.alloc(rows * 4 * 4).ptr, ctx.alloc(rows * 5 * 4).ptr, rows, H, E, 4, 1e-6, H, 0)
        ctx.dispatch_multi([A.make_op(A.OP_MOE_ROUTER, args)])
        ok = np.arange(rows) != bad
        h64 = h[ok].astype(np.float64)
        want_x = h64 / np.sqrt((h64 * h64).mean(axis=1, keepdims=True) + 1e-6) * gamma
        every = np.vstack([router, shared]).astype(np.float64)
        got_x, got = xn.read(np.float32, rows * H).reshape(rows, H), logits.read(np.float32, rows * (E + 1)).reshape(rows, E + 1)
        assert np.abs(got_x[ok] - want_x).max() <= 1e-6 * np.abs(want_x).max()
        bound = 26 * 2.0 ** -24 * 5 * np.sqrt((want_x * want_x) @ (every * every).T)
        n = E + 1 if gate else E
        want = (want_x @ every.T)[:, :n]
        assert (np.abs(got[ok][:, :n] - want) <= bound[:, :n]).all()
        rms = np.sqrt(((got[ok][:, :n] - want) ** 2).mean() / (want ** 2).mean()) * 2.0 ** 24
        assert rms <= 2.63 or (E, rows) == (512, 385)  # one row past the float32 forms
        assert gate or (got[:, E] == -7.0).all()
        assert not np.isfinite(got[bad, :n]).any()
    finally:
        ctx.destroy()


@pytest.mark.parametrize("rows", [49, 56, 64])
def test_passes_of_one_group(rows):
    """Projections and router on either side of these kernels' gap: the same bounds hold in it."""
    test_rows_of_a_pass(300, 2048, rows)
    test_router_of_a_lower_pass(rows, 512, True)


@pytest.mark.parametrize("n,k,rows", [(96, 2048, 9), (2048, 4096, 16), (70, 2048, 65), (2048, 4096, 192), (300, 2048, 512)])
def test_sums_past_binary16(n, k, rows):
    """Every activation is a binary16 number, the sum of a sub-block's 32 is not (65504 is the largest): the min term's sums are
    float32.  The bound is on what the two terms of a row add up, which cancel here: 16 ulp of float32, a fourth of what 64 roundings
    in a row could make."""
    rng = np.random.default_rng(n + rows)
    ctx = A.Context(0)
    try:
        w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
        wq = O.quantize_q4k(w)
        w64 = O.dequant_q4k(wq, k).astype(np.float64)
        x = (rng.standard_normal((rows, k)) * 500.0 + 3000.0 * np.where(np.arange(rows) % 2, 1.0, -1.0)[:, None]).astype(np.float32)
        x[rows // 2] *= 1e-4  # and a row of ordinary size among them
        assert np.abs(x.reshape(rows, -1, 32).sum(axis=2)).max() > 65504 and np.abs(x).max() < 65504
        dy = ctx.alloc(rows * n * 4)
        ctx.gemv_q4k(ctx.upload(wq), ctx.upload(x), dy, n, k, n_tok=rows)
        got, x64 = dy.read(np.float32, rows * n).reshape(rows, n), x.astype(np.float64)
        size = np.abs(x64) @ (np.abs(w64) + 2 * np.abs(w64).max(axis=1, keepdims=True)).T
        assert np.isfinite(got).all()
        assert (np.abs(got - x64 @ w64.T) <= 2.0 ** -20 * size).all()
    finally:
        ctx.destroy()
