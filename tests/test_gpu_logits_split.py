"""The output layer's product on a prepared fp32 matrix beyond 32 columns (csrc/zr_logits.hip): edges of its 32-row blocks, its tiles
of one to six 32-column blocks with four or eight waves (test_rules_cpu.py holds that the sizes here take each), and its steps of 32 k.
Tolerance: the products of 32 k are six exact terms each, added one after another in fp32 -- twelve instructions, each rounding
a partial sum at most once for every product it adds -- and the steps' sums are added in turn: at most K + 12 roundings of
2^-24 of the sum of the terms' magnitudes; the three terms left out are below one more."""
import numpy as np
import pytest

from test_gpu_backward import ctx_get
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def operands(V, H, n):
    r = np.random.default_rng(V + 100 * H + n)
    D = np.asfortranarray(r.uniform(-0.5, 0.5, (V, H)).astype(np.float32))
    return D, r.uniform(-1, 1, V).astype(np.float32), np.asfortranarray(r.uniform(-1, 1, (H, n)).astype(np.float32))


def logits_and_blocks(ctx, D, b, h):
    V, H, n = D.shape[0], D.shape[1], h.shape[1]
    blocks, off = (V + 31) // 32, (V * n + 3) // 4 * 4
    dD = ctx.array(D)
    ctx.softmax_prepare(dD, V, H)
    out = ctx.array(np.full(off + 2 * blocks * n + 1, 7.0, np.float32))
    ctx.softmax_forward(dD, ctx.array(b), V, H, ctx.array(h), n, capi.ZR_SOFTMAX_LOGITS_BLOCKS, out)
    ctx.sync()
    ctx.softmax_release(dD)
    o = out.get()
    assert o[-1] == 7.0
    return o[:V * n].reshape((V, n), order="F"), o[off:-1].reshape((n, blocks, 2))


def bound(D, b, h):
    return (D.shape[1] + 13) * 2.0 ** -24 * (np.abs(D).astype(np.float64) @ np.abs(h) + np.abs(b)[:, None])


SIZES = [(33, 1, 33), (31, 31, 64), (129, 32, 65), (257, 33, 96), (1000, 63, 97), (1000, 65, 257), (4001, 100, 160), (2049, 129, 700),
         (9001, 37, 1100), (30011, 500, 37), (33333, 64, 128), (50001, 96, 192), (8191, 300, 320), (12345, 1000, 40),
         # the tiles that none of these takes, and matrices of 64 MiB and more, whose loads have the streaming hint, with rows left over
         (2996, 64, 963), (4493, 64, 901), (11978, 64, 963), (18964, 64, 777), (16469, 64, 901), (16801, 1000, 33), (33601, 500, 97)]


@pytest.mark.parametrize("V,H,n", SIZES)
def test_logits_and_block_pairs(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    x, pairs = logits_and_blocks(ctx, D, b, h)
    want = D.astype(np.float64) @ h + b[:, None]
    assert np.all(np.abs(x - want) <= bound(D, b, h))
    pad = np.full(((V + 31) // 32 * 32, n), -np.inf)
    pad[:V] = x
    pad = pad.reshape((-1, 32, n))
    assert np.array_equal(pairs[:, :, 0].T, pad.max(1).astype(np.float32))
    s = np.exp(pad - pad.max(1, keepdims=True)).sum(1)
    # 32 terms: their additions and the exponential's argument of size up to the block's range, 2^-24 each
    assert np.all(np.abs(pairs[:, :, 1].T / s - 1.0) < (32 + 4 * np.abs(want).max()) * 2.0 ** -24)


def test_infinities_and_nan(ctx):
    V, H, n = 1000, 100, 70
    D, b, h = operands(V, H, n)
    want, most = D.astype(np.float64) @ h + b[:, None], bound(D, b, h)
    D[5, 17], D[999, 99], D[700, 3], D[130, 44] = np.inf, -np.inf, np.nan, 3.4e38  # the last rounds to infinity in bf16
    h[44] *= 1e-3
    h[17, 9], h[60, 30] = 0.0, np.inf
    x, _ = logits_and_blocks(ctx, D, b, h)
    with np.errstate(invalid="ignore"):
        want = D.astype(np.float64) @ h + b[:, None]
        most = bound(np.where(np.isfinite(D), D, 0.0), b, np.where(np.isfinite(h), h, 0.0))
    assert np.array_equal(np.isnan(x), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(x[inf], want[inf].astype(np.float32))
    fine = np.isfinite(want)
    assert np.all(np.abs(x[fine] - want[fine]) <= most[fine])


def test_decoder_width_is_the_same_with_and_without_static_scratch(ctx):
    V, H, n = 5000, 264, 100
    D, b, h = operands(V, H, n)
    dD, db, dh, x, y = ctx.array(D), ctx.array(b), ctx.array(h), ctx.empty((V, n)), ctx.empty((V, n))
    ctx.softmax_prepare(dD, V, H)
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_PROB, x)
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_PROB, y, static=True)
    ctx.sync()
    assert np.array_equal(x.get(), y.get())


@pytest.mark.parametrize("n", [33, 64, 100, 257])
def test_matrices_past_32_bit_offsets(ctx, n):
    """From 4 GiB on the row-range kernel and, beyond 256 columns, the split product take a prepared matrix."""
    V, H = 262177, 4104
    r = np.random.default_rng(n)
    dD, b = ctx.empty((V, H)), r.uniform(-1, 1, V).astype(np.float32)
    ctx.uniform_fill(7, n, dD, V * H)
    h = np.asfortranarray(r.uniform(-0.1, 0.1, (H, n)).astype(np.float32))
    out = ctx.empty((V, n))
    ctx.softmax_prepare(dD, V, H)
    try:
        ctx.softmax_forward(dD, ctx.array(b), V, H, ctx.array(h), n, capi.ZR_SOFTMAX_LOGPROB, out)
        ctx.sync()
    finally:
        ctx.softmax_release(dD)
    x = out.get()
    rows = np.r_[0:24, V // 2:V // 2 + 24, V - 24:V]
    D = np.stack([np.concatenate([ctx_get(ctx, dD.at(k * V + int(i)), (24,)) for i in rows[::24]]) for k in range(H)], axis=1)
    want, most = D.astype(np.float64) @ h + b[rows, None], bound(D, b[rows], h)
    # log-probabilities: the logits less one number a column, whose own rounding and the subtraction's are 2^-23 of it
    less = np.median(want - x[rows], axis=0)
    assert np.all(np.abs(want - x[rows] - less) <= 2 * most + 2.0 ** -23 * np.abs(less))
    assert np.all(np.abs(np.exp(x.astype(np.float64)).sum(0) - 1.0) < 1e-3)
