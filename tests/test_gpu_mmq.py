"""Token-block Q8_0 x Q8_0 products on the matrix cores, through the C ABI.

The reference runs every token through the Q8 matvec
(fortai_gguf_runtime.f90:424-465).  Bars: the per-token quantization and
the int32 block dots bit-exact against the oracle; the lane-order product
(mmq_exact, the prefill's default) bit-identical to the oracle's AVX2 matvec
of every token; the whole-block product (mmq, the fast variant) within 1e-5
relative of it (the north star allows 1e-3).
"""

import ctypes

import numpy as np
import pytest

from fortai_amd import backend as B
from fortai_amd import synth

pytestmark = pytest.mark.gpu

REL = 1e-3


def rel_err(got, want):
    want = np.asarray(want, dtype=np.float64)
    got = np.asarray(got, dtype=np.float64)
    scale = np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2)) + 1e-30)
    return float(np.max(np.abs(got - want) / scale))


def tokens_layout(ctx, buf, tokens, width):
    """Split an X8 buffer into q [blocks][tokens][32] and s [blocks][tokens]."""
    ld = (tokens + 127) // 128 * 128
    bp = (width // 32 + 3) // 4 * 4
    raw = buf.download(np.uint8, ld * bp * 36)
    q = raw[: ld * bp * 32].view(np.int8).reshape(bp, ld, 32)
    s = raw[ld * bp * 32:].view(np.float32).reshape(bp, ld)
    return q, s, ld, bp


@pytest.mark.parametrize("rows,width,tokens", [(13, 96, 5), (200, 1024, 37), (3584, 1024, 64), (1024, 3584, 70)])
def test_mmq_block_dots_and_outputs(ctx, oracle, rows, width, tokens):
    rng = np.random.default_rng(rows * 31 + width + tokens)
    w = synth.q8_blocks(rng, rows, width)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    x[0, :32] = 0.0  # an all-zero block
    nb = width // 32
    W = B.Q8Weights(ctx, w, rows, width)
    dx = ctx.upload_array(x)
    nbytes = B.load().fortai_hip_q8_tokens_bytes(tokens, width)
    dq = ctx.alloc(nbytes)
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, dq.ptr)
    q, s, ld, bp = tokens_layout(ctx, dq, tokens, width)
    # quantization: each token as the reference quantizer, zero padding
    for t in range(tokens):
        qr, sr = oracle.quantize(x[t])
        qr = qr.reshape(nb, 34)[:, 2:]
        assert np.array_equal(q[:nb, t], qr)
        assert np.array_equal(s[:nb, t].view(np.uint32), sr.view(np.uint32))
    assert not q[:, tokens:].any() and not s[:, tokens:].any()
    assert not q[nb:].any() and not s[nb:].any()
    # exact int32 block dots
    dd = ctx.alloc(tokens * rows * nb * 4)
    ctx.call("fortai_hip_q8_mmq_block_dots", ctx.h, W.h, dq.ptr, tokens, dd.ptr)
    dots = dd.download(np.int32).reshape(tokens, rows, nb)
    for t in range(tokens):
        qr, _ = oracle.quantize(x[t])
        assert np.array_equal(dots[t], oracle.block_dots(w, qr, rows, nb)), f"token {t}"
    # fp32 outputs against the reference matvec of every token; then the
    # residual epilogue in place
    out = ctx.alloc(tokens * rows * 4)
    ms = ctypes.c_float()
    ctx.call("fortai_hip_q8_mmq_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, None, ctypes.byref(ms))
    got = out.download(np.float32).reshape(tokens, rows)
    want = np.stack([oracle.matvec(w, rows, width, x[t]) for t in range(tokens)])
    assert rel_err(got, want) <= REL
    assert rel_err(got, want) <= 1e-5  # the block dots are exact: only fp32 rounding differs
    resid = rng.standard_normal((tokens, rows)).astype(np.float32)
    dr = ctx.upload_array(resid)
    ctx.call("fortai_hip_q8_mmq_device", ctx.h, W.h, dq.ptr, tokens, dr.ptr, dr.ptr, None)
    got2 = dr.download(np.float32).reshape(tokens, rows)
    assert np.array_equal(got2, (got + resid).astype(np.float32))
    W.free()


def test_mmq_prefill_shape(ctx, oracle):
    """A 4B FFN gate shape (9216 x 2560) over 512 tokens; the oracle checks a
    sample of tokens (size-independent: every token's row vector is its own
    matvec)."""
    rows, width, tokens = 9216, 2560, 512
    rng = np.random.default_rng(5)
    w = synth.q8_blocks(rng, rows, width)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    W = B.Q8Weights(ctx, w, rows, width)
    dx = ctx.upload_array(x)
    dq = ctx.alloc(B.load().fortai_hip_q8_tokens_bytes(tokens, width))
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, dq.ptr)
    out = ctx.alloc(tokens * rows * 4)
    ctx.call("fortai_hip_q8_mmq_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, None, None)
    got = out.download(np.float32).reshape(tokens, rows)
    for t in (0, 1, 63, 64, 255, 511):
        assert rel_err(got[t], oracle.matvec(w, rows, width, x[t])) <= 1e-5, f"token {t}"
    W.free()


@pytest.mark.parametrize("rows,width,tokens", [(13, 96, 5), (200, 1024, 37), (88, 256, 21), (3584, 1024, 64),
                                               (1024, 3584, 70), (9216, 2560, 130)])
def test_mmq_lane_order_bit_identical(ctx, oracle, rows, width, tokens):
    """q8_mmq_exact_kernel: every output equals the reference matvec of its
    token bit for bit (ragged rows, in the first or the second 16-row half of
    a wave's rows, partial token tiles, a 4B FFN shape); the
    residual epilogue adds in place."""
    rng = np.random.default_rng(rows + 7 * width + tokens)
    w = synth.q8_blocks(rng, rows, width)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    x[0, :32] = 0.0
    x[1 % tokens, 32:64] = 1e4
    W = B.Q8Weights(ctx, w, rows, width)
    dx = ctx.upload_array(x)
    dq = ctx.alloc(B.load().fortai_hip_q8_tokens_bytes(tokens, width))
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, dq.ptr)
    out = ctx.alloc(tokens * rows * 4)
    ctx.call("fortai_hip_q8_mmq_exact_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, None, None)
    got = out.download(np.float32).reshape(tokens, rows)
    sample = range(tokens) if tokens <= 70 else (0, 1, 63, 64, 65, 127, 128, 129)
    for t in sample:
        want = oracle.matvec(w, rows, width, x[t])
        assert np.array_equal(got[t].view(np.uint32), want.view(np.uint32)), \
            f"token {t}: max rel {rel_err(got[t], want):.2e}"
    resid = rng.standard_normal((tokens, rows)).astype(np.float32)
    dr = ctx.upload_array(resid)
    ctx.call("fortai_hip_q8_mmq_exact_device", ctx.h, W.h, dq.ptr, tokens, dr.ptr, dr.ptr, None)
    assert np.array_equal(dr.download(np.float32).reshape(tokens, rows), (got + resid).astype(np.float32))
    W.free()


@pytest.mark.parametrize("rows,width,tokens", [(1, 32, 1), (32, 128, 16), (33, 640, 17), (224, 512, 33), (225, 544, 31),
                                               (264, 1664, 48), (300, 96, 260), (17, 2560, 300), (2560, 1056, 150),
                                               (4100, 160, 200), (2100, 96, 900)])
def test_mmq_lane_order_tiles(ctx, rows, width, tokens):
    """The token product's tile choices -- 64 x 64, 32 rows x 16 and x 32
    tokens, fewer and more than eight row tiles, ragged rows and tokens, whole
    and partial groups of four chunks -- against the batched matvec of the same
    tokens (itself checked against the oracle), bit for bit, with and without
    the residual."""
    rng = np.random.default_rng(rows + 3 * width + tokens)
    W = B.Q8Weights(ctx, synth.q8_blocks(rng, rows, width), rows, width)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    x[tokens // 2, :32] = 0.0
    dx = ctx.upload_array(x)
    dq = ctx.alloc(B.load().fortai_hip_q8_tokens_bytes(tokens, width))
    out, want = ctx.alloc(tokens * rows * 4), ctx.alloc(tokens * rows * 4)
    for t in range(0, tokens, 8):
        ctx.call("fortai_hip_q8_batch_matvec_device", ctx.h, W.h, dx.ptr.value + t * width * 4, min(8, tokens - t),
                 want.ptr.value + t * rows * 4, None)
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, dq.ptr)
    ctx.call("fortai_hip_q8_mmq_exact_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, None, None)
    expect = want.download(np.float32)
    assert np.array_equal(out.download(np.float32).view(np.uint32), expect.view(np.uint32))
    resid = rng.standard_normal(tokens * rows).astype(np.float32)
    out.upload(resid)
    ctx.call("fortai_hip_q8_mmq_exact_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, out.ptr, None)
    assert np.array_equal(out.download(np.float32).view(np.uint32), (expect + resid).view(np.uint32))
    for b in (dx, dq, out, want):
        b.free()
    W.free()


def fma32(a, b, c):
    """float32 fma(a, b, c), b an integer below 2^20: the product is exact in
    float64, and the sum is rounded to odd there (its error by TwoSum; 53 >=
    2 x 24 + 2 bits), so that its rounding to float32 is the only one."""
    p, c = a.astype(np.float64) * b, c.astype(np.float64)
    s = p + c
    bb = s - p
    err = (p - (s - bb)) + (c - bb)
    even = (s.view(np.uint64) & np.uint64(1)) == 0
    odd = np.where((err != 0) & even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
    return odd.astype(np.float32)


@pytest.mark.parametrize("rows,width,tokens", [(1, 32, 1), (31, 96, 33), (130, 160, 64), (897, 288, 31), (1030, 1056, 40),
                                               (2560, 544, 700), (128, 2560, 129), (4100, 128, 520)])
def test_mmq_tiles(ctx, oracle, rows, width, tokens):
    """The whole-block product's tile choices (128 x 128 and 128 rows x 32
    tokens, fewer and more than eight row tiles, odd chunk counts): every output
    is the scalar reference's block-order sum acc = fma(w_scale * x_scale,
    dot, acc) of exact int32 block dots, bit for bit on a sample of tokens; the
    residual is added in place."""
    rng = np.random.default_rng(rows + 5 * width + tokens)
    w = synth.q8_blocks(rng, rows, width)
    nb = width // 32
    W = B.Q8Weights(ctx, w, rows, width)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    x[0, :32] = 0.0
    dx = ctx.upload_array(x)
    dq = ctx.alloc(B.load().fortai_hip_q8_tokens_bytes(tokens, width))
    out = ctx.alloc(tokens * rows * 4)
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, dq.ptr)
    ctx.call("fortai_hip_q8_mmq_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, None, None)
    got = out.download(np.float32).reshape(tokens, rows)
    ws = w.reshape(rows, nb, 34)[:, :, :2].copy().view(np.float16).reshape(rows, nb).astype(np.float32)
    for t in sorted({0, 1 % tokens, 31 % tokens, 32 % tokens, tokens // 2, tokens - 1}):
        qr, sr = oracle.quantize(x[t])
        dots = oracle.block_dots(w, qr, rows, nb).astype(np.float64)
        acc = np.zeros(rows, np.float32)
        for b in range(nb):
            acc = fma32(ws[:, b] * np.float32(sr[b]), dots[:, b], acc)
        assert np.array_equal(got[t].view(np.uint32), acc.view(np.uint32)), f"token {t}"
    resid = rng.standard_normal((tokens, rows)).astype(np.float32)
    out.upload(resid)
    ctx.call("fortai_hip_q8_mmq_device", ctx.h, W.h, dq.ptr, tokens, out.ptr, out.ptr, None)
    assert np.array_equal(out.download(np.float32).reshape(tokens, rows), (got + resid).astype(np.float32))
    for b in (dx, dq, out):
        b.free()
    W.free()


@pytest.mark.parametrize("exact", [0, 1])
@pytest.mark.parametrize("rows,width,tokens", [(1, 32, 1), (33, 640, 17), (225, 544, 31), (264, 1664, 48), (897, 288, 31),
                                               (1030, 1056, 40), (300, 96, 260), (2560, 544, 700), (2560, 1056, 150),
                                               (4100, 128, 520), (2100, 96, 900)])
def test_mmq_chunk_major_tokens(ctx, rows, width, tokens, exact):
    """Both products over the prefill's chunk-major tokens (one and several row
    tiles of every kind, ragged rows and tokens, whole and partial groups of
    chunks) give the bits of the block-major ones, with and without the
    residual, whatever the rows past the tokens hold."""
    rng = np.random.default_rng(rows + 11 * width + tokens)
    W = B.Q8Weights(ctx, synth.q8_blocks(rng, rows, width), rows, width)
    dx = ctx.upload_array(rng.standard_normal((tokens, width)).astype(np.float32))
    nbytes = B.load().fortai_hip_q8_tokens_bytes(tokens, width)
    blocks, chunks = ctx.alloc(nbytes), ctx.alloc(nbytes)
    want, got = ctx.alloc(tokens * rows * 4), ctx.alloc(tokens * rows * 4)
    ctx.call("fortai_hip_q8_quantize_tokens_device", ctx.h, dx.ptr, tokens, width, blocks.ptr)
    q, s, ld, bp = tokens_layout(ctx, blocks, tokens, width)
    cq = q.reshape(bp // 4, 4, ld, 8, 4).transpose(0, 2, 3, 1, 4).copy()
    cs = s.reshape(bp // 4, 4, ld).transpose(0, 2, 1).copy()
    cq[:, tokens:], cs[:, tokens:] = -128, np.nan
    chunks.upload(np.concatenate([cq.view(np.uint8).ravel(), cs.view(np.uint8).ravel()]))
    entry = "fortai_hip_q8_mmq_exact_device" if exact else "fortai_hip_q8_mmq_device"
    resid = rng.standard_normal(tokens * rows).astype(np.float32)
    try:
        for r in (None, resid):
            if r is not None:
                want.upload(r)
                got.upload(r)
            at = lambda b: None if r is None else b.ptr
            ctx.call(entry, ctx.h, W.h, blocks.ptr, tokens, want.ptr, at(want), None)
            ctx.call("fortai_hip_q8_mmq_chunks_device", ctx.h, W.h, chunks.ptr, tokens, exact, got.ptr, at(got))
            assert np.array_equal(got.download(np.uint32), want.download(np.uint32))
    finally:
        for b in (dx, blocks, chunks, want, got, W):
            b.free()
