"""The expert kernels that stream short per-expert lists (csrc/moe_lists.hip) against the per-(token, slot) kernels, on lists
whose lengths are the edges of what a wave takes at a time."""
import numpy as np
import pytest

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


def block(rig, topk, grouped, packed):
    c, E, _, banks = rig
    T, U = topk.shape
    rng = np.random.default_rng(T)
    xn, res = rng.standard_normal((T, H)).astype(np.float32), rng.standard_normal((T, H)).astype(np.float32)
    wts = rng.random((T, U + 1)).astype(np.float32)
    bufs = [c.upload(a) for a in (xn, topk, wts, res)]
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
