"""One LSTM node on bf16 weights and 8-row tiles (csrc/zr_lstm_rows_bf16.hip): each tile width, half k-groups (H % 32 == 16), fewer k-groups than
waves, ragged columns, both numbers of terms, hand-over of h as terms between the layers of a step.
Reference: 64 bits on the rounded weights and on the activations' own terms, so the products are exact and only the fp32 sums
differ: at most K * terms + 24 roundings of 2^-24 of the sum of the magnitudes.  A gate moves by at most that (slopes up to 1), c by the
gates' errors times |c_prev| <= 1 and |gate| <= 1, h by c's and its own gate's: four times the bound, and a few ulp of the gates' functions."""
import numpy as np
import pytest

from gpu_util import Layer, round_bf16, run_lstm_step
from zoph_rnn_amd import capi, synth

pytestmark = pytest.mark.gpu

SIZES = [(16, 1, True), (16, 40, False), (48, 33, True), (144, 17, True), (496, 65, False), (528, 20, True), (560, 48, False), (624, 33, True),
         (1008, 128, True), (1024, 64, False), (1104, 80, True), (1360, 81, False), (2000, 17, True), (2032, 63, False)]


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def terms_of(x, n):
    hi = round_bf16(x)
    return hi.astype(np.float64) + (round_bf16(x - hi) if n == 2 else 0.0)


def sigmoid(z):
    return 1.0 / (1.0 + np.exp(-z))


def node(ly, x, hp, cp, ht, mask, n):
    z, mag = [], 0.0
    for g in range(4):
        parts = [(ly["M"][g], x), (ly["Wh"][g], hp)] + ([(ly["Q"][g], ht)] if ht is not None else [])
        z.append(sum(w.astype(np.float64) @ terms_of(a, n) for w, a in parts) + ly["b"][g].reshape(-1, 1))
        mag = np.maximum(mag, sum(np.abs(w).astype(np.float64) @ np.abs(a) for w, a in parts) + np.abs(ly["b"][g]).reshape(-1, 1))
    i, f, c_, o = sigmoid(z[0]), sigmoid(z[1]), np.tanh(z[2]), sigmoid(z[3])
    c = f * cp + i * c_
    H = x.shape[0]
    bound = 4 * ((3 * H * n + 24) * 2.0 ** -24 * mag + 2.0 ** -21)
    return {"i": i, "f": f, "c_tilde": c_, "o": o, "c": c * mask, "h": o * np.tanh(c) * mask}, bound


def weights(g, H, feed):
    ly = synth.lstm_layer(g, H, feed_input=feed)
    for k in ("M", "Wh") + (("Q",) if feed else ()):
        ly[k] = [np.asfortranarray(round_bf16(m)) for m in ly[k]]
    return ly


@pytest.mark.parametrize("n", [2, 1])
@pytest.mark.parametrize("H,mb,feed", SIZES)
def test_node(ctx, H, mb, feed, n):
    g = synth.rng(171, H + mb)
    ly = weights(g, H, feed)
    x, hp, cp = (synth.uniform(g, (H, mb), -1, 1) for _ in range(3))
    ht = synth.uniform(g, (H, mb), -1, 1) if feed else None
    mask = (g.random(mb) > 0.2).astype(np.int32)
    layer = Layer(ctx, ly, bf16=True)
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, n)
    try:
        got = run_lstm_step(ctx, layer, x, hp, cp, mask, htild=ht, want_gates=True)
    finally:
        ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, 2)
        layer.close()
    want, bound = node(ly, x, hp, cp, ht, mask, n)
    for k, v in want.items():
        assert np.all(np.abs(got[k] - v) <= bound), (k, np.max(np.abs(got[k] - v) / bound))


@pytest.mark.parametrize("n", [2, 1])
@pytest.mark.parametrize("H,mb", [(48, 5), (624, 33), (1040, 70)])
def test_step_of_three_layers(ctx, H, mb, n):
    g = synth.rng(172, H + mb)
    lys = [weights(g, H, l == 0) for l in range(3)]
    V = 50
    embed, ids = synth.uniform(g, (H, V), -1, 1), g.integers(0, V, mb).astype(np.int32)
    hp, cp = [synth.uniform(g, (H, mb), -1, 1) for _ in lys], [synth.uniform(g, (H, mb), -1, 1) for _ in lys]
    ht, mask = synth.uniform(g, (H, mb), -1, 1), np.ones(mb, np.int32)
    layers = [Layer(ctx, ly, bf16=True) for ly in lys]
    h, c = [ctx.empty((H, mb)) for _ in lys], [ctx.empty((H, mb)) for _ in lys]
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, n)
    try:
        ctx.lstm_decoder_step([ly.w for ly in layers], ctx.array(embed), V, ctx.array(ids), [ctx.array(a) for a in hp], [ctx.array(a) for a in cp],
                              ctx.array(mask), mb, h, c, d_htild=ctx.array(ht))
        ctx.sync()
    finally:
        ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, 2)
        for ly in layers:
            ly.close()
    x = np.asfortranarray(embed[:, ids])
    for l, ly in enumerate(lys):  # each layer from the h that the one below it left
        want, bound = node(ly, x, hp[l], cp[l], ht if l == 0 else None, mask, n)
        x = h[l].get()
        assert np.all(np.abs(x - want["h"]) <= bound) and np.all(np.abs(c[l].get() - want["c"]) <= bound)
