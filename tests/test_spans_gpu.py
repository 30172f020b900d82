"""shv_copy_spans and shv_upload_words: what they leave in memory, at the edges of their launches."""
import ctypes as C

import numpy as np
import pytest

import shv

pytestmark = pytest.mark.gpu
A = shv.api


@pytest.fixture(scope="module")
def ctx():
    c = A.Context()
    yield c
    c.destroy()


# one span, spans of every length around a step of the kernel (64 KB x 8), more spans than a launch lists (128), addresses
# and lengths that are only whole words
@pytest.mark.parametrize("n_spans,lengths,skew", [(1, (16,), 0), (3, (4, 65536, 524288 + 16), 0), (130, (48,), 0), (129, (20, 4096, 12), 4), (5, (0, 64), 8)])
def test_copy_spans(ctx, n_spans, lengths, skew):
    rng = np.random.default_rng(n_spans)
    sizes = [lengths[i % len(lengths)] for i in range(n_spans)]
    total = sum(s + 32 for s in sizes) + 64
    src, before = rng.integers(0, 256, total).astype(np.uint8), rng.integers(0, 256, total).astype(np.uint8)
    d_src, d_dst = ctx.upload(src), ctx.upload(before)
    want, at, spans = before.copy(), 0, []
    for i, s in enumerate(sizes):
        at += skew
        zero = i % 3 == 1
        spans.append(A.Span(d_dst.at(at), None if zero else d_src.at(at), s))
        want[at:at + s] = 0 if zero else src[at:at + s]
        at = (at + s + 31) // 16 * 16
    A.check(ctx.L.shv_copy_spans(ctx.h, (A.Span * n_spans)(*spans), n_spans))
    assert np.array_equal(d_dst.read(np.uint8, total), want)


@pytest.mark.parametrize("counts", [(1,), (640,), (641, 3), (0, 5, 2000), tuple([2] * 70)])
def test_upload_words(ctx, counts):
    rng = np.random.default_rng(len(counts))
    before = rng.integers(0, 1 << 30, sum(counts) + 2 * len(counts) + 1).astype(np.int32)
    dst, want, at = ctx.upload(before), before.copy(), 1
    arrays, words = [], []
    for n in counts:
        v = rng.integers(0, 1 << 30, max(n, 1)).astype(np.int32)[:n]
        arrays.append(v)
        words.append(A.Words(dst.at(at * 4), v.ctypes.data, n))
        want[at:at + n] = v
        at += n + 2
    A.check(ctx.L.shv_upload_words(ctx.h, (A.Words * len(words))(*words), len(words)))
    for v in arrays:
        v[:] = -1  # the words have left the caller's memory
    assert np.array_equal(dst.read(np.int32, len(before)), want)


def test_spans_and_words_refuse_what_they_cannot_do(ctx):
    b = ctx.alloc(64)
    for span in (A.Span(b.at(2), None, 4), A.Span(b.ptr, b.at(32), 6), A.Span(None, b.ptr, 4)):
        with pytest.raises(A.ShvError):
            A.check(ctx.L.shv_copy_spans(ctx.h, C.byref(span), 1))
    v = np.zeros(4, np.int32)
    for w in (A.Words(None, v.ctypes.data, 4), A.Words(b.ptr, None, 4), A.Words(b.at(2), v.ctypes.data, 1)):
        with pytest.raises(A.ShvError):
            A.check(ctx.L.shv_upload_words(ctx.h, C.byref(w), 1))


def test_blocks_no_context_owns(ctx):
    p = C.c_void_p()
    hbm = ctx.props().hbm_bytes
    assert ctx.L.shv_block_alloc(0, 1 << 20, hbm, C.byref(p)) == -3 and p.value is None  # would leave less than all of it
    A.check(ctx.L.shv_block_alloc(0, 1 << 20, hbm // 16, C.byref(p)))
    want = np.random.default_rng(1).integers(0, 256, 1 << 20).astype(np.uint8)
    A.check(ctx.L.shv_upload(ctx.h, p, want.ctypes.data, want.nbytes))
    got = np.zeros_like(want)
    A.check(ctx.L.shv_block_read(0, got.ctypes.data, p, got.nbytes))
    assert np.array_equal(got, want)
    A.check(ctx.L.shv_block_free(0, p))
