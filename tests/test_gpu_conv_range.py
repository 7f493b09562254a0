"""The conv kernel's two passes: products of fp32 operands as fp16 parts for the outputs whose sums
are large enough beside what the parts round off, from the fp32 operands for every other output.

The bar on values is componentwise, |err| <= c n 2^-24 sum |w x| over the n products of an output
(float64 reference): an fp32 sum in any order keeps to it with c = 1, the parts add n/2 + 8 of the
same.  It holds at every input scale and for any mix of magnitudes, among the inputs of an output and
among the weights of a row.  Which pass an output comes from depends on its own inputs and its rows'
weights, so a column that does not see a disturbance keeps its bits."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle_lib as ol
from conftest import load_package
from test_gpu_conv import gpu_conv, gpu_convT
from test_gpu_decoder import relerr, say

pkg = load_package()
synth = pkg.synth
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = pkg.Ctx(arena_mb=512)
    yield c
    c.close()


def conv64(x, W, b, pad, dil, stride):
    """float64 conv of x [B][cin][T]: (values, sum of |products|)"""
    cout, cin, K = W.shape
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pad, pad)))
    n = (xp.shape[-1] - dil * (K - 1) - 1) // stride + 1
    y = np.zeros((len(x), cout, n))
    a = np.zeros_like(y)
    for k in range(K):
        cols = xp[:, :, k * dil:k * dil + (n - 1) * stride + 1:stride]
        y += np.matmul(W[:, :, k].astype(np.float64), cols)
        a += np.matmul(np.abs(W[:, :, k].astype(np.float64)), np.abs(cols))
    return y + b.astype(np.float64)[:, None], a


def case(cin, cout, K, T, seed=0, B=1):
    rng = np.random.default_rng(seed + 1000 * K + cin)
    x = rng.standard_normal((B, cin, T)).astype(np.float32)
    W = (rng.standard_normal((cout, cin, K)) / np.sqrt(cin * K)).astype(np.float32)
    return rng, x, W, (0.1 * rng.standard_normal(cout)).astype(np.float32)


# cin (20: channel padding, 16 / 64: whole chunks), K (5: the rolled loop), dilation, stride
SHAPES = [(64, 3, 1, 1), (64, 7, 3, 1), (64, 11, 5, 1), (64, 5, 2, 1), (20, 3, 1, 1), (16, 7, 1, 2)]


@pytest.mark.parametrize("cin,K,dil,stride", SHAPES)
@pytest.mark.parametrize("scale", [2.0 ** -100, 1e-6, 2.0 ** -9, 1.0, 300.0, 2e3, 1e30])
def test_every_input_scale_meets_the_fp32_bound(ctx, cin, K, dil, stride, scale):
    rng, x, W, b = case(cin, 40, K, 150)
    x *= np.float32(scale)
    b *= np.float32(scale)
    pad = (K - 1) * dil // 2
    y = gpu_conv(ctx, x, synth.pack_conv(W), b, 40, K, stride, pad, dil)
    ref, mag = conv64(x, W, b, pad, dil, stride)
    bound = (cin * K + 2) * 2.0 ** -24 * (mag + np.abs(b.astype(np.float64))[:, None])
    assert np.all(np.abs(y[:, :40] - ref) <= bound)


@pytest.mark.parametrize("cin,K,dil,stride", SHAPES)
@pytest.mark.parametrize("value", [5e4, np.inf, -np.inf, np.nan, -3.4028235e38])
def test_a_disturbed_column_keeps_to_itself(ctx, cin, K, dil, stride, value):
    """One input far out of range: the outputs that see it are what an fp32 conv gives, every other
    output keeps its bits (in the same tile and in the neighbouring ones)."""
    rng, x, W, b = case(cin, 40, K, 260, B=2)
    wp, pad = synth.pack_conv(W), (K - 1) * dil // 2
    y0 = gpu_conv(ctx, x, wp, b, 40, K, stride, pad, dil)[:, :40]
    t = 101
    x[1, cin // 2, t] = value
    y = gpu_conv(ctx, x, wp, b, 40, K, stride, pad, dil)[:, :40]
    n = y.shape[-1]
    sees = np.zeros(n, bool)
    for k in range(K):
        q = t + pad - k * dil
        if q % stride == 0 and 0 <= q // stride < n:
            sees[q // stride] = True
    assert sees.any() and not sees.all()
    assert np.array_equal(y[0], y0[0]) and np.array_equal(y[1][:, ~sees], y0[1][:, ~sees])
    with np.errstate(invalid="ignore", over="ignore"):
        ref, mag = conv64(x, W, b, pad, dil, stride)
    got, want = y[1][:, sees], ref[1][:, sees]
    if np.isnan(value):
        assert np.all(np.isnan(got))
    elif np.isinf(value):
        assert np.array_equal(got, np.where(np.isfinite(want), got, want)) and not np.any(np.isfinite(got))
    else:
        bound = (cin * K + 2) * 2.0 ** -24 * (mag[1][:, sees] + 1.0)
        assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("bad", [np.inf, np.nan, 2.0 ** -110, 1e30, 0.0])
def test_weight_rows_without_an_fp16_form(ctx, bad):
    """A row with an inf or NaN weight, one far below 2^-100, a huge one, a zero one: that row is what
    an fp32 conv gives and the rows of other blocks keep their bits."""
    rng, x, W, b = case(48, 96, 7, 130)
    y0 = gpu_conv(ctx, x, synth.pack_conv(W), b, 96, 7, 1, 3, 1)
    row = 37
    if np.isfinite(bad):
        W[row] = (np.float32(bad) * rng.standard_normal(W[row].shape)).astype(np.float32)
        b[row] = 0.0
    else:
        W[row, 5, 2] = bad
    y = gpu_conv(ctx, x, synth.pack_conv(W), b, 96, 7, 1, 3, 1)
    other = np.r_[0:32, 64:96]
    assert np.array_equal(y[:, other], y0[:, other])
    ref, mag = conv64(x, W, b, 3, 1, 1) if np.isfinite(bad) else (None, None)
    if np.isfinite(bad):
        assert np.all(np.abs(y[:, row] - ref[:, row]) <= (48 * 7 + 2) * 2.0 ** -24 * mag[:, row])
        rest = np.delete(np.arange(96), row)
        assert np.all(np.abs(y - ref)[:, rest] <= (48 * 7 + 2) * 2.0 ** -24 * (mag[:, rest] + 1.0))
    else:   # columns 2 .. see the weight; tap 2 reads column t - 1: all but the first
        assert not np.any(np.isfinite(y[:, row, 1:])) and np.all(np.isfinite(y[:, np.delete(np.arange(96), row)]))


@pytest.mark.parametrize("scale", [1e-7, 1.0, 2e3])
def test_convT_input_scales(ctx, scale):
    rng = np.random.default_rng(5)
    x = (scale * rng.standard_normal((1, 64, 61))).astype(np.float32)
    W = (rng.standard_normal((64, 32, 16)) / 16).astype(np.float32)
    b = (scale * rng.standard_normal(32)).astype(np.float32)
    wp = synth.pack_convtranspose(W, 4)
    y, ref = gpu_convT(ctx, x, wp, b, 32, 16, 4, 6), ol.convT(x, wp, b, 32, 16, 4, 6)
    assert relerr(y, ref) < 1e-4


@pytest.mark.parametrize("scale", [1e-7, 3e3])
def test_decoder_stages_out_of_range(scale):
    """Latents (and biases) that leave every activation far out of the fp16 parts' range: each stage
    of the decode, whose convs read split planes, against the oracle at the per-layer bar."""
    say(f"decoder stages at scale {scale}")
    ctx = pkg.Ctx(arena_mb=256)
    ws, bs = synth.decoder_weights(77)
    bs = [np.float32(scale) * b for b in bs]
    model = pkg.Model(ctx, ws, bs)
    T = 19
    z = np.float32(scale) * synth.latent(T, 3)
    ref, rst = ol.decoder(ws, bs, z, stages=True)
    dz, dw = pkg.DevBuf.of(ctx, z), pkg.DevBuf(256 * T)
    st = [pkg.DevBuf(r.size) for r in rst]
    arr = (C.c_void_p * 6)(*[s.ptr for s in st])
    assert ctx.lib.ptd_decode_stages(ctx.ptr, model.ptr, dz.ptr, T, dw.ptr, arr) == 0
    for i, (s, r) in enumerate(zip(st, rst)):
        e = relerr(s.download(ctx).reshape(r.shape), r)
        say(f"  stage {i}: {e:.3g}")
        assert e < 1e-4, i
    for d in [dz, dw] + st:
        d.free()
    model.close()
    ctx.close()


def test_layer_alone_equals_layer_in_a_decode():
    """ptd_layer splits its fp32 input itself, the decode's convs read split planes their producers
    wrote: the same bits (conv_pre -> ups.0, through the stage tensors)."""
    ctx = pkg.Ctx(arena_mb=256)
    ws, bs = synth.decoder_weights(1234)
    model = pkg.Model(ctx, ws, bs)
    T = 45
    dz, dw = pkg.DevBuf.of(ctx, synth.latent(T, 8)), pkg.DevBuf(256 * T)
    h, x0, y = pkg.DevBuf(512 * T), pkg.DevBuf(256 * 4 * T), pkg.DevBuf(256 * 4 * T)
    arr = (C.c_void_p * 6)(h.ptr, x0.ptr, None, None, None, None)
    assert ctx.lib.ptd_decode_stages(ctx.ptr, model.ptr, dz.ptr, T, dw.ptr, arr) == 0
    assert ctx.lib.ptd_layer(ctx.ptr, model.ptr, 1, h.ptr, T, 1, y.ptr, 0.0, 0.0) == 0
    assert np.array_equal(y.download(ctx), x0.download(ctx))
    for d in (dz, dw, h, x0, y):
        d.free()
    model.close()
    ctx.close()


# mixes of magnitudes: inputs by channel, weights by element, weights that undo the inputs' scales,
# and rows that select one quiet channel beside loud ones
def _mixed(kind, rng, x, W):
    cout, cin, K = W.shape
    if kind == "inputs":
        return x * 10.0 ** rng.uniform(-30, 3, (cin, 1)), W
    if kind == "weights":
        return x, W * 10.0 ** rng.uniform(-12, 6, W.shape)
    if kind == "opposed":
        s = 10.0 ** rng.uniform(-8, 3, (cin, 1))
        return x / s, W * s
    W = np.zeros_like(W)
    for m in range(cout):
        W[m, (5 * m) % cin, m % K] = 1.0
        if m % 4 == 1:
            W[m, (5 * m + 1) % cin, m % K] = 1e-6   # beside a weight far below the row's largest
    return x * 10.0 ** rng.uniform(-14, 2, (cin, 1)), W


@pytest.mark.parametrize("cin,K,dil,stride", SHAPES)
@pytest.mark.parametrize("kind", ["inputs", "weights", "opposed", "select"])
@pytest.mark.parametrize("split,nb", [(0, 0), (2, 1), (2, 2), (4, 1), (4, 2)])
def test_mixed_magnitudes_meet_the_componentwise_bound(ctx, cin, K, dil, stride, kind, split, nb, knob_env):
    """|err| <= (n + n/2 + 9) 2^-24 sum |w x|, n the nonzero weights of the row: the sum's own rounding
    and the bias, and the parts'.  On every tile shape."""
    if split:
        knob_env.setenv("PTK_CONV_SPLIT", str(split))
        knob_env.setenv("PTK_CONV_NB", str(nb))
    rng, x, W, _ = case(cin, 72, K, 150, seed=7)
    x, W = _mixed(kind, rng, x, W)
    x, W, b = x.astype(np.float32), W.astype(np.float32), np.zeros(72, np.float32)
    pad = (K - 1) * dil // 2
    y = gpu_conv(ctx, x, synth.pack_conv(W), b, 72, K, stride, pad, dil)[:, :72]
    ref, mag = conv64(x, W, b, pad, dil, stride)
    n = np.count_nonzero(W, axis=(1, 2))[:, None]
    tiny = n * 2.0 ** -149   # products below fp32's range
    assert np.all(np.abs(y - ref) <= (1.5 * n + 9) * 2.0 ** -24 * mag + tiny)


def test_examples_of_lost_range(ctx):
    """One quiet input beside a loud one, one small weight beside a large one: exactly what fp32 gives
    (a product with 1 is exact)."""
    for q in (1e-6, 1e-7, 1e-10, 1e-30):
        x = np.zeros((1, 16, 40), np.float32)
        x[:, 0], x[:, 1] = 1.0, np.float32(q)
        W = np.zeros((32, 16, 1), np.float32)
        W[:, 1] = 1.0
        y = gpu_conv(ctx, x, synth.pack_conv(W), np.zeros(32, np.float32), 32, 1, 1, 0, 1)
        assert np.all(np.abs(y - np.float32(q)) <= 2.0 ** -21 * q), q
    x[:, 1], W[:, 0], W[:, 1] = 1.1e-6, 1e-6, 1e6
    y = gpu_conv(ctx, x, synth.pack_conv(W), np.zeros(32, np.float32), 32, 1, 1, 0, 1)
    want = np.float64(np.float32(1e-6)) + np.float64(np.float32(1e6)) * np.float64(np.float32(1.1e-6))
    assert np.all(np.abs(y - want) <= 12 * 2.0 ** -24 * want)


def _stats(ctx):
    n = (C.c_uint64 * 2)()
    assert ctx.lib.ptd_debug_conv_stats(n) == 0
    return np.array([n[0], n[1]])


def test_ordinary_inputs_and_silence_stay_on_the_first_pass(ctx):
    """N(0, 1) inputs leave no output to the second pass; columns of zeros, alone and next to sound,
    leave theirs and find nothing to compute again: the bias, exactly."""
    rng, x, W, b = case(192, 96, 7, 400, seed=3)
    wp = synth.pack_conv(W)
    n0 = _stats(ctx)
    y0 = gpu_conv(ctx, x, wp, b, 96, 7, 1, 3, 1)
    n1 = _stats(ctx)
    assert not np.any(n1 - n0)
    x[:, :, 100:300] = 0.0
    y = gpu_conv(ctx, x, wp, b, 96, 7, 1, 3, 1)
    n2 = _stats(ctx)
    assert n2[0] > n1[0] and n2[1] == n1[1]
    assert np.array_equal(y[:, :, 103:297], np.broadcast_to(b[:, None], y[:, :, 103:297].shape))
    assert np.array_equal(y[:, :, :97], y0[:, :, :97]) and np.array_equal(y[:, :, 303:], y0[:, :, 303:])
    x[0, 17, 200] = 1e-30   # below the parts' range: the second pass sees it
    y = gpu_conv(ctx, x, wp, np.zeros(96, np.float32), 96, 7, 1, 3, 1)
    assert _stats(ctx)[1] > n2[1]
    want = np.float64(W[:, 17, ::-1]) * np.float64(x[0, 17, 200])
    assert np.all(np.abs(y[0, :, 197:204] - want) <= 2.0 ** -23 * np.abs(want))


@pytest.mark.parametrize("cout", [30, 37, 62, 70, 97])
@pytest.mark.parametrize("nb", [1, 2])
def test_rows_of_a_partial_block(ctx, cout, nb, knob_env):
    """Outputs that do not fill their last block of 32 rows, nor its last group of four: bias and
    LeakyReLU of the ones that exist, and nothing behind them is written over (batch 2: the rows of the
    next item follow)."""
    knob_env.setenv("PTK_CONV_NB", str(nb))
    rng, x, W, b = case(48, cout, 7, 133, seed=11, B=2)
    y = gpu_conv(ctx, x, synth.pack_conv(W), b, cout, 7, 1, 3, 1)
    ref, mag = conv64(x, W, b, 3, 1, 1)
    bound = (48 * 7 * 1.5 + 9) * 2.0 ** -24 * (mag + np.abs(b.astype(np.float64))[:, None])
    assert np.all(np.abs(y[:, :cout] - ref) <= bound)
