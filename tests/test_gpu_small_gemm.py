"""Small products on narrow tiles (csrc/zr_small_gemm.hip): sizes at the edges of the 16 x 16, 16 x 32 and 32 x 32 tiles, of the
groups of 16 k that the eight waves take in turn and of the groups a wave has in flight, in every operand layout, of one segment and of
several or grouped (test_rules_cpu.py holds that the sizes here reach every tile, depth and layout that the rule gives out).
Tolerance: K products summed one after another in fp32 are off by at most K 2^-24 times the sum of their magnitudes; twelve
more for the waves' sums and what is added to them."""
import numpy as np
import pytest

from gpu_util import round_bf16
from test_gpu_error_products import run as backward
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def check(got, a, b, extra=0.0):
    want = a.astype(np.float64) @ b.astype(np.float64) + extra
    assert np.all(np.abs(got - want) <= (a.shape[1] + 12) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b) + np.abs(extra)))
    return want


SIZES = [(1, 1, 16), (15, 17, 17), (16, 16, 19), (17, 15, 31), (33, 1, 128), (64, 64, 129), (100, 20, 100), (100, 20, 257), (31, 300, 383), (500, 37, 500),
         (777, 130, 777), (1000, 128, 1000), (129, 33, 513), (300, 200, 1025), (2000, 128, 2000), (65, 250, 4001),
         (430, 230, 90)]


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_plain_operands(ctx, M, N, K, trans):
    r = np.random.default_rng(M + 1000 * N + K)
    a, b = r.uniform(-1, 1, (M, K)).astype(np.float32), r.uniform(-1, 1, (K, N)).astype(np.float32)
    lda, ldb, ldc = (K if trans else M) + 3, K + 1, M + 2  # odd leading dimensions: no operand is 16-byte aligned throughout
    A = np.full((lda, M if trans else K), np.nan, np.float32, order="F")
    A[:K if trans else M] = a.T if trans else a
    B = np.full((ldb, N), np.nan, np.float32, order="F")
    B[:K] = b
    dC, dA, dB = ctx.array(np.full((ldc, N), 7.0, np.float32, order="F")), ctx.array(A), ctx.array(B)
    ctx.gemm(trans, M, N, K, dA, lda, dB, ldb, dC, ldc)
    ctx.sync()
    got = dC.get()
    want = check(got[:M], a, b)
    assert np.all(got[M:] == 7.0)
    # nothing stands in for k past the end beside an infinity, and a NaN reaches its own row only
    A[(K - 1, M - 1) if trans else (M - 1, K - 1)] = np.inf
    A[(0, 0)] = np.nan
    dA.set(A)
    ctx.gemm(trans, M, N, K, dA, lda, dB, ldb, dC, ldc)
    ctx.sync()
    got = dC.get()[:M]
    rest = np.ones(M, bool)
    rest[[0, M - 1]] = False
    assert np.isnan(got[0]).all() and np.all(np.abs(got[rest] - want[rest]) <= (K + 12) * 2.0 ** -24 * (np.abs(a[rest]).astype(np.float64) @ np.abs(b)))
    if M > 1:
        assert np.array_equal(np.sign(got[M - 1]), np.sign(b[K - 1])) and np.isinf(got[M - 1]).all()


FEED = [(16, 1), (17, 3), (20, 20), (100, 33), (333, 17), (500, 64), (1000, 128), (257, 241), (513, 241)]


@pytest.mark.parametrize("H,mb", FEED)
def test_four_segments(ctx, H, mb):
    """The feed-input error, sum over the gates of Q_g^T d_g, in one launch."""
    r = np.random.default_rng(7 * H + mb)
    Q = [np.asfortranarray(r.uniform(-1, 1, (H, H)).astype(np.float32)) for _ in range(4)]
    dg, ht = np.asfortranarray(r.uniform(-1, 1, (4 * H, mb)).astype(np.float32)), np.zeros((H, mb), np.float32, order="F")
    d_Q, d_dg, d_ht, d_err, d_dQ = [ctx.array(q) for q in Q], ctx.array(dg), ctx.array(ht), ctx.empty((H, mb)), ctx.zeros((4 * H, H))
    ctx.lstm_feed_backward(d_Q, H, mb, d_dg, d_ht, d_err, d_dQ)
    ctx.sync()
    check(d_err.get(), np.concatenate([q.T for q in Q], 1), dg)


BF16 = [(16, 1, 2), (48, 37, 1), (48, 37, 2), (112, 256, 2), (512, 64, 1), (1024, 64, 2), (1024, 128, 1)]


@pytest.mark.parametrize("H,mb,terms", BF16)
def test_bf16_output_product(ctx, H, mb, terms):
    """h~ = tanh(W_c1 c + W_c2 h + b) of the attention step on bf16 matrices, the context as the step gives it."""
    r = np.random.default_rng(11 * H + mb)
    S, D = 6, 2
    W = [np.asfortranarray(r.uniform(-0.2, 0.2, (H, H)).astype(np.float32)) for _ in range(4)]
    vp, bias = r.uniform(-0.2, 0.2, H).astype(np.float32), r.uniform(-0.2, 0.2, H).astype(np.float32)
    hs = np.asfortranarray(r.uniform(-1, 1, (H, S * mb)).astype(np.float32))
    h = np.asfortranarray(r.uniform(-1, 1, (H, mb)).astype(np.float32))
    d_W, d_v, d_b, d_hs, d_h = [ctx.array(w) for w in W], ctx.array(vp), ctx.array(bias), ctx.array(hs), ctx.array(h)
    a = ctx.attn_create(H, mb, D, d_W[0], d_W[1], d_v, d_b, d_W[2], d_W[3], [d_hs.at(t * H * mb) for t in range(S)])
    ctx.attn_use_bf16_weights(a)
    info, mask = ctx.array(np.r_[np.full(mb, S), np.zeros(mb)].astype(np.int32)), ctx.array(np.ones(mb, np.int32))
    d_ht, d_c = ctx.empty((H, mb)), ctx.empty((H, mb))
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, terms)
    ctx.attn_step(a, info, d_h, mask, d_ht, d_ctx=d_c)
    ctx.sync()
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, 2)
    ctx.attn_destroy(a)
    x = np.concatenate([d_c.get(), h])
    hi = round_bf16(x)
    x = hi.astype(np.float64) + (round_bf16(x - hi) if terms == 2 else 0.0)
    w = round_bf16(np.concatenate([W[2], W[3]], 1)).astype(np.float64)
    want = np.tanh(w @ x + bias[:, None])
    # sums of 2H (two terms: 4H) products and the tanh's own rounding
    assert np.all(np.abs(d_ht.get() - want) <= (2 * terms * H + 12) * 2.0 ** -24 * (np.abs(w) @ np.abs(x) + np.abs(bias[:, None])) + 2.0 ** -22)


# fp32 matrices as they lie (0) or prepared (1), bf16 ones (2), with one and with two terms an activation
ATTENTION = [(H, mb, 1, 2) for H, mb in [(16, 1), (136, 1), (264, 1), (129, 226), (264, 241), (257, 241), (272, 241), (520, 37), (52, 19), (333, 130)]] + \
    [(H, mb, 2, terms) for terms in (1, 2)
     for H, mb in [(16, 1), (272, 1), (528, 1), (1040, 1), (144, 226), (272, 241), (400, 163), (528, 241), (784, 33)]] + [(52, 19, 0, 2), (17, 3, 0, 2)]


@pytest.mark.parametrize("H,mb,layout,terms", ATTENTION)
def test_attention_step(ctx, H, mb, layout, terms):
    """All products of an attention step: W_p h through p_t, W_a^T h through the alignments (with the p_t of the step), W_c1 c + W_c2 h (with
    its context) as h~.  A part of 2^-20 is for exponentials, tanh and sums over five source states."""
    r = np.random.default_rng(13 * H + mb)
    S, D = 5, 6
    W = [np.asfortranarray(r.uniform(-0.2, 0.2, (H, H)).astype(np.float32)) for _ in range(4)]
    vp, bias = r.uniform(-0.2, 0.2, H).astype(np.float32), r.uniform(-0.2, 0.2, H).astype(np.float32)
    hs = [np.asfortranarray((r.uniform(-1, 1, (H, mb)) / np.sqrt(H)).astype(np.float32)) for _ in range(S)]
    h = np.asfortranarray(r.uniform(-1, 1, (H, mb)).astype(np.float32))
    d_W, d_v, d_b, d_hs, d_h = [ctx.array(w) for w in W], ctx.array(vp), ctx.array(bias), [ctx.array(x) for x in hs], ctx.array(h)
    a = ctx.attn_create(H, mb, D, d_W[0], d_W[1], d_v, d_b, d_W[2], d_W[3], d_hs)
    if layout == 2:
        ctx.attn_use_bf16_weights(a)
    elif layout == 1:
        ctx.attn_prepare(a)
    info, mask = ctx.array(np.r_[np.full(mb, S), np.zeros(mb)].astype(np.int32)), ctx.array(np.ones(mb, np.int32))
    d_ht, d_c, d_p, d_al, d_ix = ctx.empty((H, mb)), ctx.empty((H, mb)), ctx.empty((mb,)), ctx.empty((mb, 2 * D + 1)), ctx.empty((mb, 2 * D + 1), np.int32)
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, terms)
    ctx.set_option(capi.ZR_OPT_ATTN_SINGLE_LAUNCH, 1)
    ctx.attn_step(a, info, d_h, mask, d_ht, d_al, d_ix, d_p, d_c)
    ctx.sync()
    ctx.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, 2)
    ctx.set_option(capi.ZR_OPT_ATTN_SINGLE_LAUNCH, 0)
    ctx.attn_destroy(a)

    def product(w, x):  # 64 bits, and how far a sum in fp32 may be off
        w, x = w.astype(np.float64), x.astype(np.float64)
        if layout == 2:
            w, hi = round_bf16(w.astype(np.float32)).astype(np.float64), round_bf16(x.astype(np.float32))
            x = hi.astype(np.float64) + (round_bf16((x - hi).astype(np.float32)) if terms == 2 else 0.0)
        return w @ x, ((terms if layout == 2 else 1) * w.shape[1] + 12) * 2.0 ** -24 * (np.abs(w) @ np.abs(x))
    Wa, Wp, Wc1, Wc2 = W
    pre, off = product(Wp, h)
    p = S / (1.0 + np.exp(-(vp.astype(np.float64) @ np.tanh(pre))))
    assert np.all(np.abs(d_p.get() - p) <= S * 0.25 * (np.abs(vp) @ off + (H + 12) * 2.0 ** -24 * np.abs(vp).sum()) + S * 2.0 ** -20)
    q, off = product(Wa.T, h)
    x = np.stack(hs).astype(np.float64)
    score, off = np.einsum("shb,hb->sb", x, q), np.einsum("shb,hb->sb", np.abs(x), off + (H + 12) * 2.0 ** -24 * np.abs(q))
    e = np.exp(score - np.maximum(score.max(0), 0.0))
    place = np.arange(S)[:, None]  # source position s is state S - 1 - s
    want = (e / e.sum(0))[::-1] * np.exp(-(d_p.get().astype(np.float64) - place) ** 2 / (2 * (D * D / 4.0)))
    got = d_al.get().T
    assert np.array_equal(d_ix.get().T[:S], np.repeat(place, mb, 1))
    assert np.all(np.abs(got[:S] / want - 1.0) <= 2.1 * off.max(0) + 2.0 ** -20)
    z1, off1 = product(Wc1, d_c.get())
    z2, off2 = product(Wc2, h)
    assert np.all(np.abs(d_ht.get() - np.tanh(z1 + z2 + bias[:, None])) <= off1 + off2 + 2.0 ** -20)


# layers, H, columns: the products of a full diagonal, on k-interleaved operands (H a multiple of four) and as they lie
DIAGONALS = [(1, 16, 1), (1, 68, 1), (1, 132, 1), (8, 20, 130), (7, 100, 33), (8, 36, 163), (1, 17, 1), (1, 65, 1), (1, 129, 1), (8, 17, 130), (7, 97, 33)]


@pytest.mark.parametrize("L,H,mb", DIAGONALS)
def test_grouped(ctx, L, H, mb):
    M, Wh, d, eh, below = backward(ctx, L, H, mb, lambda r, T: r.standard_normal((T, mb, H)))
    for got, W, dg in [(eh[l], Wh[l], d[l][0]) for l in range(L)] + [(below[t], M[0], d[0][t]) for t in range(L)]:
        check(got, np.concatenate(W, axis=0).T, dg)
