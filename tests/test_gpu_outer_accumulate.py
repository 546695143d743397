"""The weight gradients of a single node, C += A B^T over the minibatch, on the kernel that reads both operands as they lie:
zr_lstm_feed_backward's (4H x H) and, two at a time, zr_attn_backward's (H x H, tests/test_gpu_backward.py holds their
values).  Sizes at the edges of its 32 x 32 tiles, of its rounds of 32 columns and of its range (96 columns for the smaller H,
256 from H = 274 on), beyond which the transposing products serve.
Tolerance: K products summed one after another in fp32 and added to C are off by at most (K + 2) 2^-24 times the sum of the
terms' magnitudes; the product instruction may add its two k at a time, which is not more."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("H,mb", [(8, 1), (9, 2), (8, 31), (31, 32), (33, 33), (63, 64), (65, 65), (100, 8), (129, 255), (300, 20),
                                  (64, 256), (64, 257), (500, 64), (1000, 128), (64, 96), (64, 97), (274, 255), (275, 256), (300, 257)])
def test_feed_gradient_against_64_bits(ctx, H, mb):
    r = np.random.default_rng(1000 * H + mb)
    Q = [np.asfortranarray(r.uniform(-0.08, 0.08, (H, H)).astype(np.float32)) for _ in range(4)]
    dg = np.asfortranarray(r.standard_normal((4 * H, mb)).astype(np.float32))
    ht = np.asfortranarray(np.tanh(r.standard_normal((H, mb))).astype(np.float32))
    dQ0 = np.asfortranarray(r.standard_normal((4 * H, H)).astype(np.float32))
    d_dQ, d_err = ctx.array(dQ0), ctx.empty((H, mb))
    d_Q, d_dg, d_ht = [ctx.array(q) for q in Q], ctx.array(dg), ctx.array(ht)
    ctx.lstm_feed_backward(d_Q, H, mb, d_dg, d_ht, d_err, d_dQ)
    ctx.sync()
    want = dQ0.astype(np.float64) + dg.astype(np.float64) @ ht.astype(np.float64).T
    bound = (mb + 2) * 2.0 ** -24 * (np.abs(dQ0) + np.abs(dg).astype(np.float64) @ np.abs(ht).T)
    assert np.all(np.abs(d_dQ.get() - want) <= bound)
    # an infinite error reaches its own row only
    dg[0, mb - 1] = np.inf
    d_dg.set(dg)
    d_dQ.set(dQ0)
    ctx.lstm_feed_backward(d_Q, H, mb, d_dg, d_ht, d_err, d_dQ)
    ctx.sync()
    got = d_dQ.get()
    assert not np.isfinite(got[0]).any() and np.all(np.abs(got[1:] - want[1:]) <= bound[1:])


@pytest.mark.parametrize("H,mb", [(64, 96), (300, 128), (500, 256), (1000, 200)])
def test_feed_gradient_is_rounded_in_short_chains(ctx, H, mb):
    """Four sums of a quarter of the products each, not one of all.  An addition rounds its result by a relative 2^-23 / sqrt(12)
    * 0.73 = 2.5e-8 in the 2-norm (mantissas spread evenly in their logarithm); the n partial sums of a chain have
    half the final square on average, and independent roundings add in squares: sqrt(n / 2) of them, n = mb / 4, and three for
    the chains' sum.  A quarter above that passes (measured 5 % above); one chain would be twice it."""
    r = np.random.default_rng(2000 * H + mb)
    Q = [np.zeros((H, H), np.float32, order="F") for _ in range(4)]
    dg = np.asfortranarray(r.uniform(-1, 1, (4 * H, mb)).astype(np.float32))
    ht = np.asfortranarray(r.uniform(-1, 1, (H, mb)).astype(np.float32))
    d_dQ = ctx.zeros((4 * H, H))
    d_Q, d_dg, d_ht, d_err = [ctx.array(q) for q in Q], ctx.array(dg), ctx.array(ht), ctx.empty((H, mb))
    ctx.lstm_feed_backward(d_Q, H, mb, d_dg, d_ht, d_err, d_dQ)
    ctx.sync()
    want = dg.astype(np.float64) @ ht.astype(np.float64).T
    error = np.linalg.norm(d_dQ.get() - want) / np.linalg.norm(want)
    assert error < 1.25 * 2.5e-8 * np.sqrt(mb / 8 + 3)
