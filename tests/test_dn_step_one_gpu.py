"""One row of each sequence (dn_step_one_kernel) against the first of two rows through the kernel of several: the same numbers, bit
for bit.  Positions whose history starts before the sequence, wraps the ring or lies inside it; up to three sequences and from four
on (two and four state rows a wave); slots out of order; one state plane written in place, or a plane kept beside the committed one."""
import numpy as np
import pytest

import shv

pytestmark = pytest.mark.gpu
A = shv.api
HK, HV, D, SLOTS, RING = 2, 4, 128, 13, 8
W = 2 * HK * D + 2 * HV * D + 2 * HV


@pytest.mark.parametrize("n_seq", [1, 3, 4, 12])
@pytest.mark.parametrize("planes", [1, 3])
def test_first_row(ctx, n_seq, planes):
    rng = np.random.default_rng(100 * planes + n_seq)
    ring = rng.standard_normal((SLOTS, RING, W)).astype(np.float32)
    state = (rng.standard_normal((SLOTS, planes, HV, D, D)) * 0.1).astype(np.float32)
    conv = (rng.standard_normal((2 * HK * D + HV * D, 4)) * 0.3).astype(np.float32)
    a, dt = (-np.exp(rng.standard_normal(HV))).astype(np.float32), rng.standard_normal(HV).astype(np.float32)
    slot = rng.permutation(SLOTS)[:n_seq].astype(np.int32)
    pos = np.resize([0, 1, 2, 9, 7, 12], n_seq).astype(np.int32)
    cur = rng.integers(0, 3, size=SLOTS).astype(np.int32)
    bufs = [ctx.upload(v) for v in (ring, conv, a, dt, pos, slot, cur)]
    p = [b.ptr for b in bufs]

    def step(rows, n_planes, states):
        d_state, d_out = ctx.upload(states), ctx.alloc(n_seq * rows * HV * D * 4)
        args = A.DnStepArgs(p[0], p[1], p[2], p[3], d_state.ptr, d_out.ptr, p[4], p[5], n_seq, rows, HK, HV, D, 4, RING, W, 1e-6, 0,
                            p[6], n_planes, 1 if n_planes > 1 else 0, None, 0)
        ctx.dispatch_multi([A.make_op(A.OP_DN_STEP, args)])
        got = d_state.read(np.float32, states.size).reshape(states.shape), d_out.read(np.float32, n_seq * rows * HV * D).reshape(n_seq, rows, HV * D)
        d_state.free()
        d_out.free()
        return got

    # two rows, every prefix's state kept, from the committed copy
    kept = np.zeros((SLOTS, 3, HV, D, D), np.float32)
    at = cur % 3
    kept[np.arange(SLOTS), at] = state[:, 0] if planes == 1 else state[np.arange(SLOTS), at]
    want_state, want_out = step(2, 3, kept)
    got_state, got_out = step(1, planes, state)
    assert np.array_equal(got_out[:, 0], want_out[:, 0])
    for s in range(SLOTS):
        new = got_state[s, 0 if planes == 1 else (at[s] + 1) % 3]
        if s in slot:
            assert np.array_equal(new, want_state[s, (at[s] + 1) % 3]), s
        else:
            assert np.array_equal(got_state[s], state[s]), s
    for b in bufs:
        b.free()
