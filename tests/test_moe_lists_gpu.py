"""The expert kernels that stream short per-expert lists (csrc/moe_lists.hip) against the per-(token, slot) kernels, on lists
whose lengths are the edges of what a wave takes at a time, and against float64 where activations or their sums leave binary16."""
import numpy as np
import pytest

import oracle_lib as O
import shv

pytestmark = pytest.mark.gpu
A = shv.api
H, F = 2048, 512


@pytest.fixture(scope="module")
def rig():
    c = A.Context()
    E = 24
    rng = np.random.default_rng(5)

    def bank(rows, k, seed):
        src, dst = c.alloc(rows * k * 4), c.alloc(rows * k // 256 * 144)
        import ctypes as C
        A.check(c.L.shv_fill_normal(c.h, C.byref(A.FillNormalArgs(src.ptr, rows * k, seed, 0.0, 0.02, 0))))
        A.check(c.L.shv_quantize_q4k(c.h, C.byref(A.QuantizeQ4KArgs(src.ptr, dst.ptr, rows, k))))
        c.sync()
        src.free()
        return dst

    banks = [bank(E * F, H, 1), bank(E * F, H, 2), bank(E * H, F, 3), bank(F, H, 4), bank(F, H, 5), bank(H, F, 6)]
    yield c, E, rng, banks
    c.destroy()


def selection(lengths, used, rng):
    """A table [tokens][used] of distinct experts a token, expert e chosen lengths[e] times."""
    total = sum(lengths)
    assert total % used == 0
    tokens = total // used
    assert max(lengths) <= tokens
    # expert after expert down the columns: an expert's run is no longer than a column, so no token sees it twice
    flat = np.concatenate([np.full(n, e) for e, n in enumerate(lengths)]).reshape(used, tokens).T
    return np.ascontiguousarray(flat[rng.permutation(tokens)], dtype=np.int32)


def block(rig, topk, grouped, packed, order=slice(None)):
    c, E, _, banks = rig
    T, U = topk.shape
    rng = np.random.default_rng(T)
    xn, res = rng.standard_normal((T, H)).astype(np.float32), rng.standard_normal((T, H)).astype(np.float32)
    wts = rng.random((T, U + 1)).astype(np.float32)
    bufs = [c.upload(a[order]) for a in (xn, topk, wts, res)]
    act, out = c.alloc(T * (U + 1) * F * 4), c.alloc(T * H * 4)
    group, pairs = c.alloc((2 * E + 1 + T * U) * 4), c.alloc(T * (U + 1) * H * 4)
    g, u, d, gs, us, ds = (b.ptr for b in banks)
    ua = A.MoeUpArgs(bufs[0].ptr, bufs[1].ptr, g, u, gs, us, act.ptr, T, H, U, F, None, None, E, 0, 0, 0, 0, group.ptr if grouped else None, 0, packed)
    da = A.MoeDownArgs(act.ptr, bufs[1].ptr, bufs[2].ptr, d, ds, bufs[3].ptr, out.ptr, T, H, U, F, H, H, 0, 0, E,
                       group.ptr if grouped else None, pairs.ptr if grouped else None, 1 if grouped else 0, packed)
    c.dispatch_multi([A.make_op(A.OP_MOE_UP, ua), A.make_op(A.OP_MOE_DOWN, da)])
    got = out.read(np.float32, T * H).reshape(T, H)
    for b in bufs + [act, out, group, pairs]:
        b.free()
    return got


# (lengths, used): eight tokens at a time up to six pairs an expert, sixteen up to fifteen, and on either side of the rule
@pytest.mark.parametrize("lengths,used", [
    ([0, 1, 2, 7, 8, 9, 5, 0] + [2] * 16, 1),            # 64 tokens: below the rule
    ([0, 1, 2, 7, 8, 9, 6, 0] + [2] * 16, 1),            # 65 tokens: the shortest
    ([16, 17, 33, 1, 0, 8, 9, 0] + [3] * 16, 2),         # lists of several passes of eight
    ([6] * 24, 2),                                       # 144 pairs, exactly six an expert
    ([6] * 23 + [8], 2),                                 # one more: sixteen at a time
    ([0, 1, 8, 9, 15, 16, 17, 33, 34, 47] + [12] * 13 + [14], 2),
    ([15] * 24, 4),                                      # fifteen an expert, the last of these kernels' passes
    ([15] * 23 + [18], 3),                               # past it
])
@pytest.mark.parametrize("packed", [1, 0])
def test_lists_are_the_slots(rig, lengths, used, packed):
    rng = np.random.default_rng(sum(lengths))
    topk = selection(lengths, used, rng)
    want, got = block(rig, topk, False, 0), block(rig, topk, True, packed)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= 1e-5, (topk.shape, rel)
    assert np.max(np.abs(got - want)) <= 1e-4 * np.sqrt(np.mean(want ** 2))


LENGTHS = [0, 1, 2, 7, 8, 9, 6, 0] + [2] * 16  # 65 tokens of one expert each, eight listed tokens a time
SIXTEENS = [0, 1, 8, 9, 15, 16, 17, 7] + [8] * 15 + [9]  # 202 tokens, sixteen a time


def expert_rows(rig, bank, e, rows, k):
    raw = rig[3][bank].read(np.uint8, rows * k // 256 * 144, e * rows * k // 256 * 144)
    return O.dequant_q4k(raw, k).reshape(rows, k).astype(np.float64)


def up64(x, gate, up):
    """SwiGLU of a token's gate and up products, and what rounding them once in 2^20 of their terms' sizes makes of it."""
    g, u = x @ gate.T, x @ up.T
    size = lambda w: np.abs(x) @ (np.abs(w) + 2 * np.abs(w).max(axis=1, keepdims=True)).T
    sig = 1 / (1 + np.exp(-np.clip(g, -700, 700)))
    return g * sig * u, 2.0 ** -20 * (size(gate) * np.abs(u) * 1.1 + size(up) * np.abs(g) * sig)  # |d silu| <= 1.1


@pytest.mark.parametrize("lengths", [LENGTHS, SIXTEENS])
def test_sums_past_binary16(rig, lengths):
    """Activations are binary16 numbers, a sub-block's sum of 32 is not: the min term's sums are float32."""
    c, E, _, banks = rig
    rng = np.random.default_rng(3)
    topk = selection(lengths, 1, rng)
    T = len(topk)
    xn = (rng.standard_normal((T, H)) * 500 + 3000 * np.where(np.arange(T) % 2, 1, -1)[:, None]).astype(np.float32)
    xn[T // 3] *= 1e-4
    bufs = [c.upload(a) for a in (xn, topk)]
    act, group = c.alloc(T * 2 * F * 4), c.alloc((2 * E + 1 + T) * 4)
    ua = A.MoeUpArgs(bufs[0].ptr, bufs[1].ptr, banks[0].ptr, banks[1].ptr, banks[3].ptr, banks[4].ptr, act.ptr, T, H, 1, F, None, None, E, 0, 0, 0, 0, group.ptr, 0, 0)
    c.dispatch_multi([A.make_op(A.OP_MOE_UP, ua)])
    got = act.read(np.float32, T * 2 * F).reshape(T, 2, F)
    for b in bufs + [act, group]:
        b.free()
    assert np.isfinite(got).all()
    for e in range(1, 7):
        at = np.flatnonzero(topk[:, 0] == e)
        want, tol = up64(xn[at].astype(np.float64), expert_rows(rig, 0, e, F, H), expert_rows(rig, 1, e, F, H))
        assert (np.abs(got[at, 0] - want) <= tol).all(), e
    want, tol = up64(xn.astype(np.float64), expert_rows(rig, 3, 0, F, H), expert_rows(rig, 4, 0, F, H))
    assert (np.abs(got[:, 1] - want) <= tol).all()


# act as floats from 128 rows on goes to the grouped down projection, whose operands keep binary16's range
@pytest.mark.parametrize("lengths,packed", [(LENGTHS, 1), (LENGTHS, 0), (SIXTEENS, 1)])
def test_values_of_any_size(rig, lengths, packed):
    """Rows whose activations, whose SwiGLU values or whose SwiGLU sub-blocks among one another are past binary16's range or far
    below its normal numbers, against float64: each row as exact as any other."""
    c, E, _, banks = rig
    rng = np.random.default_rng(4)
    topk = selection(lengths, 1, rng)
    T = len(topk)
    # SwiGLU goes with the square of a row's size: 1e-8 .. 1e12; from gates of some size on, half of its values are next to nothing
    xn = (rng.standard_normal((T, H)) * 10.0 ** rng.uniform(-4, 6, size=(T, 1))).astype(np.float32)
    wts = np.ones((T, 2), np.float32)
    wts[:, 1] = rng.choice([0, 1], T)  # half of the rows without the shared expert, which would hide the routed one's small values
    bufs = [c.upload(a) for a in (xn, topk, wts)]
    act, out = c.alloc(T * 2 * F * 4), c.alloc(T * H * 4)
    group, pairs = c.alloc((2 * E + 1 + T) * 4), c.alloc(T * 2 * H * 4)
    g, u, d, gs, us, ds = (b.ptr for b in banks)
    ua = A.MoeUpArgs(bufs[0].ptr, bufs[1].ptr, g, u, gs, us, act.ptr, T, H, 1, F, None, None, E, 0, 0, 0, 0, group.ptr, 0, packed)
    da = A.MoeDownArgs(act.ptr, bufs[1].ptr, bufs[2].ptr, d, ds, None, out.ptr, T, H, 1, F, H, H, 0, 0, E, group.ptr, pairs.ptr, 1, packed)
    c.dispatch_multi([A.make_op(A.OP_MOE_UP, ua), A.make_op(A.OP_MOE_DOWN, da)])
    got = out.read(np.float32, T * H).reshape(T, H)
    for b in bufs + [act, out, group, pairs]:
        b.free()
    x64 = xn.astype(np.float64)
    shared = up64(x64, expert_rows(rig, 3, 0, F, H), expert_rows(rig, 4, 0, F, H))[0] @ expert_rows(rig, 5, 0, H, F).T
    for e in range(1, 7):
        at = np.flatnonzero(topk[:, 0] == e)
        want = up64(x64[at], expert_rows(rig, 0, e, F, H), expert_rows(rig, 1, e, F, H))[0] @ expert_rows(rig, 2, e, H, F).T + wts[at, 1:] * shared[at]
        err = np.linalg.norm(got[at] - want, axis=1) / np.linalg.norm(want, axis=1)
        # three projections in a row of float32 sums, as the tests beside this one state it
        assert err.max() <= 1e-5, (e, at[err.argmax()], float(err.max()))


@pytest.mark.parametrize("T", [106, 380])  # eight listed tokens a time and sixteen; 67 and 238 pairs a block that places them: waves of one that race
def test_the_same_pass_again_is_the_same(T):
    """Lists of every length, most of them in several passes or past eight: bit for bit, from call to call."""
    c, E, U = A.Context(), 256, 10
    import ctypes as C

    def bank(rows, k, seed):
        src, dst = c.alloc(rows * k * 4), c.alloc(rows * k // 256 * 144)
        A.check(c.L.shv_fill_normal(c.h, C.byref(A.FillNormalArgs(src.ptr, rows * k, seed, 0.0, 0.02, 0))))
        A.check(c.L.shv_quantize_q4k(c.h, C.byref(A.QuantizeQ4KArgs(src.ptr, dst.ptr, rows, k))))
        c.sync()
        src.free()
        return dst

    rows, down = bank(E * F, H, 1), bank(E * H, F, 2)  # gate and up the same bank, the shared expert the first of it
    rng = np.random.default_rng(T)
    topk = np.argsort(rng.random((T, E)) * (1 + np.arange(E)), axis=1)[:, :U].astype(np.int32)
    xn, res, wts = (rng.standard_normal((T, H)).astype(np.float32) for _ in range(3))
    bufs = dx, dt, dr, dw = [c.upload(a) for a in (xn, topk, res, wts[:, :U + 1].copy())]
    act, out = c.alloc(T * (U + 1) * F * 4), c.alloc(T * H * 4)
    group, pairs = c.alloc((2 * E + 1 + T * U) * 4), c.alloc(T * (U + 1) * H * 4)
    ua = A.MoeUpArgs(dx.ptr, dt.ptr, rows.ptr, rows.ptr, rows.ptr, rows.ptr, act.ptr, T, H, U, F, None, None, E, 0, 0, 0, 0, group.ptr, 0, 1)
    da = A.MoeDownArgs(act.ptr, dt.ptr, dw.ptr, down.ptr, down.ptr, dr.ptr, out.ptr, T, H, U, F, H, H, 0, 0, E, group.ptr, pairs.ptr, 1, 1)
    first = None
    for _ in range(8):
        c.dispatch_multi([A.make_op(A.OP_MOE_UP, ua), A.make_op(A.OP_MOE_DOWN, da)])
        got, lists = out.read(np.float32, T * H), group.read(np.int32, 2 * E + 1 + T * U)
        if first is None:
            first = got, lists
            for e in range(E):
                want = np.flatnonzero((topk == e).any(axis=1))
                assert np.array_equal(lists[E + 1 + lists[e]:E + 1 + lists[e + 1]] // (U + 1), want)
        assert np.array_equal(got, first[0]) and np.array_equal(lists, first[1])
    for b in bufs + [act, out, group, pairs, rows, down]:
        b.free()
    c.destroy()


@pytest.mark.parametrize("T,E,U", [(65, 24, 1), (820, 600, 10), (896, 600, 10)])  # 65 pairs; 8200 and 8960: past a block's first 8192
def test_the_lists_themselves(T, E, U):
    """Starts, lists by token and the experts by length, made by one launch whose blocks each count every pair; experts nobody chose,
    one that every token did."""
    c, rng = A.Context(), np.random.default_rng(T)
    p = rng.random((T, E)) * (1 + np.arange(E) % 7)
    p[:, 3], p[:, 5] = 9.0, -1.0
    topk = np.argsort(-p, axis=1)[:, :U].astype(np.int32)
    bank = c.alloc(E * F * (H // 256) * 144).zero()
    act, group = c.alloc(T * (U + 1) * F * 4), c.alloc((2 * E + 1 + T * U) * 4)
    x, tk = c.upload(rng.standard_normal((T, H)).astype(np.float32)), c.upload(topk)
    c.dispatch_multi([A.make_op(A.OP_MOE_UP, A.MoeUpArgs(x.ptr, tk.ptr, bank.ptr, bank.ptr, bank.ptr, bank.ptr, act.ptr, T, H, U, F, None, None, E,
                                                         0, 0, 0, 0, group.ptr, 0, 1))])
    got = group.read(np.int32, 2 * E + 1 + T * U)
    flat = topk.ravel()
    count = np.bincount(flat, minlength=E)
    assert np.array_equal(got[:E + 1], np.concatenate([[0], np.cumsum(count)]))
    order = np.argsort(flat, kind="stable")
    assert np.array_equal(got[E + 1:E + 1 + T * U], order // U * (U + 1) + order % U)
    assert np.array_equal(got[E + 1 + T * U:], np.argsort(-count, kind="stable"))
    c.destroy()
