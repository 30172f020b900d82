"""Passes of hundreds of rows (csrc/long_tiles.hpp): projections against float64 (gemm_long.hip), expert lists around the tiles of 32, 64
and 96 rows against the per-(token, slot) kernels (moe_long.hip)."""
import numpy as np
import pytest

import oracle_lib as O
import shv
from test_moe_lists_gpu import block, expert_rows, rig, selection, up64  # noqa: F401 (rig is a fixture)

pytestmark = pytest.mark.gpu
A = shv.api
H, F = 2048, 512


@pytest.fixture(scope="module")
def ctx():
    c = A.Context(0)
    yield c
    c.destroy()


# every width; the fewest rows of each, whole and ragged groups of 64; weight rows inside a tile, a block of 128, of 256; blocks of either
# kind (256 weight rows from 2048 x 4096 of 1800 rows on, of 256 columns where 128 make more than two blocks a compute unit), in strips of eight groups and in a last one that is narrower
@pytest.mark.parametrize("n,k,rows", [(17, 256, 193), (2055, 256, 1920), (2055, 256, 2950), (300, 512, 256), (513, 1024, 449), (129, 2048, 513), (2055, 2048, 1090), (70, 4096, 577), (2048, 4096, 1801)])
def test_rows_of_a_long_pass(ctx, n, k, rows):
    """The norm folded in and the residual in place, then no prologue and a ring that wraps.  2^-17: 32 bits' sums of up to 4096 products
    in a fixed order, each product as exact as one float32."""
    rng = np.random.default_rng(n + k + rows)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    w[n // 2] = 0.015  # constant rows: a super-block whose d is zero, whose mins are not
    wq = O.quantize_q4k(w)
    w64 = O.dequant_q4k(wq, k).astype(np.float64)
    x = (rng.standard_normal((rows, k)) * 10.0 ** rng.uniform(-6, 9, size=(rows, 1))).astype(np.float32)  # the sums of 32, too, leave binary16
    x[rows // 3] = 0.0
    x[rows // 5] += 5 * np.abs(x[rows // 5]).max()
    gamma = (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    x64, res = x.astype(np.float64), rng.standard_normal((rows, n)).astype(np.float32)
    bufs = dw, dx, dg, dy = ctx.upload(wq), ctx.upload(x), ctx.upload(gamma), ctx.upload(res)
    ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_RMSNORM, gamma=dg, residual=dy)
    xn = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-6) * gamma
    want, got = xn @ w64.T + res, dy.read(np.float32, rows * n).reshape(rows, n)
    size = np.abs(xn) @ (np.abs(w64) + 2 * np.abs(w64).max(axis=1, keepdims=True)).T + np.abs(res)
    assert (np.abs(got - want) <= 2.0 ** -17 * size).all()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.sqrt(np.mean(err ** 2)) <= 1e-5, float(err.max())
    slots, pos = rows + 3, np.array([rows - 2], np.int32)
    ring, dpos = ctx.upload(np.full((slots, n), -7.0, np.float32)), ctx.upload(pos)
    ctx.gemv_q4k(dw, dx, ring, n, k, n_tok=rows, pos=dpos, seq_len=rows, ring_slots=slots, ring_stride=n)
    got, at = ring.read(np.float32, slots * n).reshape(slots, n), (pos[0] + np.arange(rows)) % slots
    want = x64 @ w64.T
    size = np.abs(x64) @ (np.abs(w64) + 2 * np.abs(w64).max(axis=1, keepdims=True)).T
    assert (np.abs(got[at] - want) <= 2.0 ** -17 * size).all() and (got[at][rows // 3] == 0).all()
    assert (np.delete(got, at, axis=0) == -7.0).all()
    for b in bufs + (ring, dpos):
        b.free()


@pytest.mark.parametrize("gate", ["ring", "rows", "heads"])
@pytest.mark.parametrize("rows", [577, 1801])
def test_gated_rows_of_a_long_pass(ctx, rows, gate):
    """The output projections' prologues: the norm of each head of 128 and the gate of a ring that wraps, or the gate of rows of its own;
    the gate beside each head of 256's queries.  2^-16: a prologue of float32 (a head's sum of squares, a square root, the gate's
    exponential: 2^-18 and less of a value each) before 2^-17 as above."""
    rng = np.random.default_rng(rows)
    n, k = 2048, 4096
    wq = O.quantize_q4k((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    w64 = O.dequant_q4k(wq, k).astype(np.float64)
    x, res = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal((rows, n)).astype(np.float32)
    x[rows // 2] *= 1e6
    x[rows // 3] *= 1e-4
    z = rng.standard_normal((rows, k)).astype(np.float32) * 3
    gamma = (1 + 0.1 * rng.standard_normal(128)).astype(np.float32)
    bufs = [ctx.upload(wq), ctx.upload(x), ctx.upload(res), ctx.upload(gamma)]
    dw, dx, dy, dg = bufs
    x64 = x.astype(np.float64)
    if gate == "heads":
        held = np.concatenate([rng.standard_normal((rows, k // 256, 256)).astype(np.float32), z.reshape(rows, k // 256, 256)], axis=2)
        bufs.append(ctx.upload(held))
        ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_MUL_SIGMOID, z=bufs[-1], head_dim=256, z_stride=2 * k, residual=dy)
    else:
        heads = x64.reshape(rows, -1, 128)
        x64 = (heads / np.sqrt((heads * heads).mean(axis=2, keepdims=True) + 1e-6) * gamma).reshape(rows, k)
        if gate == "ring":
            slots, pos = rows + 5, 2 * rows
            ring = np.full((2, slots, k + 32), np.nan, np.float32)
            ring[1, (pos + np.arange(rows)) % slots, 16:16 + k] = z
            bufs += [ctx.upload(ring), ctx.upload(np.array([pos], np.int32)), ctx.upload(np.array([1], np.int32))]
            ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_GATED_NORM, gamma=dg, z=bufs[4].at(64), head_dim=128, residual=dy,
                         pos=bufs[5], slot=bufs[6], seq_len=rows, ring_slots=slots, ring_stride=k + 32, z_ring=1)
        else:
            bufs.append(ctx.upload(z))
            ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows, prologue=A.PRO_GATED_NORM, gamma=dg, z=bufs[4], head_dim=128, residual=dy)
    x64 /= 1 + np.exp(-z.astype(np.float64))
    want, got = x64 @ w64.T + res, dy.read(np.float32, rows * n).reshape(rows, n)
    size = np.abs(x64) @ (np.abs(w64) + 2 * np.abs(w64).max(axis=1, keepdims=True)).T + np.abs(res)
    assert (np.abs(got - want) <= 2.0 ** -16 * size).all()
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.sqrt(np.mean(err ** 2)) <= 1e-5, float(err.max())
    for b in bufs:
        b.free()


def test_an_infinity_stays_in_its_row(ctx):
    n, k, rows = 96, 2048, 600
    rng = np.random.default_rng(2)
    wq = O.quantize_q4k((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[70, 5], x[71, 9] = np.inf, np.nan
    dw, dx, dy = ctx.upload(wq), ctx.upload(x), ctx.alloc(rows * n * 4)
    ctx.gemv_q4k(dw, dx, dy, n, k, n_tok=rows)
    got = dy.read(np.float32, rows * n).reshape(rows, n)
    assert not np.isfinite(got[70:72]).any()
    keep = np.delete(np.arange(rows), [70, 71])
    want = x[keep].astype(np.float64) @ O.dequant_q4k(wq, k).astype(np.float64).T
    assert np.linalg.norm(got[keep] - want) <= 1e-5 * np.linalg.norm(want)


# (lengths, used): lists on the edges of one, two and three tiles and of what a pass takes, and the shared expert's last pass of each height
@pytest.mark.parametrize("lengths,used", [
    ([0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 129, 193] + [40] * 9 + [41], 4),  # 357 tokens
    ([16] * 22 + [20, 24], 2),                                                           # 198
    ([0] + [17] * 20 + [30] * 3, 1),                                                     # 430
])
@pytest.mark.parametrize("packed", [1, 0])
def test_long_lists_are_the_slots(rig, lengths, used, packed):  # noqa: F811
    topk = selection(lengths, used, np.random.default_rng(sum(lengths)))
    want, got = block(rig, topk, False, 0), block(rig, topk, True, packed)
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= 1e-5, (topk.shape, rel)
    assert np.max(np.abs(got - want)) <= 1e-4 * np.sqrt(np.mean(want ** 2))


# walks of up to 32, 64 and 96 tokens, on either side of both lines (24 and 60 tokens an expert), lists on the edges of each
@pytest.mark.parametrize("lengths,used", [
    ([24] * 16 + [1, 31, 32, 33, 64, 6, 1, 24], 3),
    ([24] * 16 + [1, 31, 32, 33, 64, 65, 0, 2], 4),
    ([60] * 16 + [63, 64, 65, 66, 97, 95, 29, 1], 4),
    ([60] * 15 + [63, 64, 65, 96, 97, 129, 31, 32, 103], 4),
])
@pytest.mark.parametrize("packed", [1, 0])
def test_walks_of_every_height(rig, lengths, used, packed):  # noqa: F811
    test_long_lists_are_the_slots(rig, lengths, used, packed)


@pytest.mark.parametrize("packed", [1, 0])
def test_a_token_is_the_same_in_any_place_of_a_list(rig, packed):  # noqa: F811
    """A list's order is the order in which its tokens were counted, another one from call to call: a token's result must not depend on
    which pass over the list it falls to, nor on its row there.  Bit for bit, the tokens in another order and turned round."""
    topk = selection([97, 98, 101, 128, 129, 160, 193] + [40] * 16 + [42], 4, np.random.default_rng(3))
    want = block(rig, topk, True, packed)
    for order in (np.arange(len(topk))[::-1], np.random.default_rng(4).permutation(len(topk))):
        assert np.array_equal(block(rig, topk, True, packed, order), want[order])


@pytest.mark.parametrize("lengths,used", [([24] * 24, 3), ([15] * 24, 3)])  # long lists, and the list kernels'
@pytest.mark.parametrize("packed", [1, 0])
def test_act_on_a_floats_grid(rig, lengths, used, packed):  # noqa: F811
    """shv_moe_up writes act wherever a float may lie, the same bytes; operands off the sixteen-byte grid are refused by the down
    projection that would read them, and the pass after that is nobody's but its own."""
    c, E, _, banks = rig
    topk = selection(lengths, used, np.random.default_rng(5))
    T = len(topk)
    dx, dt = c.upload(np.random.default_rng(6).standard_normal((T, 2048)).astype(np.float32)), c.upload(topk)
    words = T * (used + 1) * 512
    act, group = c.upload(np.zeros(words + 4, np.float32)), c.alloc((2 * E + 1 + T * used) * 4)
    pairs, out, wts = c.alloc(T * (used + 1) * 2048 * 4), c.alloc(T * 2048 * 4), c.upload(np.ones((T, used + 1), np.float32))
    g, u, d, gs, us, ds = (b.ptr for b in banks)

    def up(at):
        c.dispatch_multi([A.make_op(A.OP_MOE_UP, A.MoeUpArgs(dx.ptr, dt.ptr, g, u, gs, us, act.ptr + at, T, 2048, used, 512, None, None, E, 0, 0, 0, 0, group.ptr, 0, packed))])
        return act.read(np.uint32, words, at)

    want = up(0)
    for at in (4, 8, 12):
        assert np.array_equal(up(at), want)
    if packed:
        with pytest.raises(A.ShvError, match="left act as matrix-core operands"):
            c.dispatch_multi([A.make_op(A.OP_MOE_DOWN, A.MoeDownArgs(act.ptr + 12, dt.ptr, wts.ptr, d, ds, None, out.ptr, T, 2048, used, 512, 2048, 2048, 0, 0, E, group.ptr, pairs.ptr, 1, 1))])
    assert np.array_equal(up(0), want)
    for b in (dx, dt, act, group, pairs, out, wts):
        b.free()


# the kernels of walks of up to one, two and three tiles, lists of all their passes
@pytest.mark.parametrize("lengths", [[17, 31, 32, 33, 1, 65] + [20] * 18, [33, 63, 64, 65, 1, 95] + [40] * 18, [97, 64, 65, 128, 193, 31] + [70] * 18])
def test_gate_and_up_of_rows_of_any_size(rig, lengths):  # noqa: F811
    """Rows whose values or whose sums of 32 are past binary16 or far below its normal numbers, against float64, each as exact as any other;
    an infinity stays in its row.  2^-18: the two projections' sums of 2048 products and their scales, each product as exact as one float32."""
    c, E, _, banks = rig
    rng = np.random.default_rng(sum(lengths))
    topk = selection(lengths, 1, rng)
    T = len(topk)
    xn = (rng.standard_normal((T, H)) * 500 + 3000 * np.where(np.arange(T) % 2, 1, -1)[:, None]) * 10.0 ** rng.uniform(-7, 5, size=(T, 1))
    xn = xn.astype(np.float32)
    lost = [int(np.flatnonzero(topk[:, 0] == 1)[4]), int(np.flatnonzero(topk[:, 0] == 3)[-1])]
    xn[lost[0], 700], xn[lost[1], 31] = np.inf, np.nan
    bufs = [c.upload(a) for a in (xn, topk)]
    act, group = c.alloc(T * 2 * F * 4), c.alloc((2 * E + 1 + T) * 4)
    ua = A.MoeUpArgs(bufs[0].ptr, bufs[1].ptr, banks[0].ptr, banks[1].ptr, banks[3].ptr, banks[4].ptr, act.ptr, T, H, 1, F, None, None, E, 0, 0, 0, 0, group.ptr, 0, 0)
    c.dispatch_multi([A.make_op(A.OP_MOE_UP, ua)])
    got = act.read(np.float32, T * 2 * F).reshape(T, 2, F)
    for b in bufs + [act, group]:
        b.free()
    assert not np.isfinite(got[lost]).any()
    kept = np.delete(np.arange(T), lost)
    assert np.isfinite(got[kept]).all()
    for e in range(E + 1):  # the last: the shared expert, whose rows are every token's
        at = np.intersect1d(kept, np.flatnonzero(topk[:, 0] == e)) if e < E else kept
        gate, up = (expert_rows(rig, 0, e, F, H), expert_rows(rig, 1, e, F, H)) if e < E else (expert_rows(rig, 3, 0, F, H), expert_rows(rig, 4, 0, F, H))
        want, tol = up64(xn[at].astype(np.float64), gate, up)
        assert (np.abs(got[at, int(e == E)] - want) <= 4 * tol).all(), (e, float(np.max(np.abs(got[at, int(e == E)] - want) / np.maximum(tol, 1e-300))))
