"""Normalising the output matrix (softmax_normalize_kernel in csrc/zr_softmax.hip): columns shorter than an access, edges of a workgroup's rows
with one, two and four accesses a thread, columns at odd addresses, the block pairs folded by every workgroup or in a launch of their own, in place and
beside the logits.  Reference: 64 bits on the logits the call leaves.  A column's sum is off by the exponentials of 32-row
blocks (argument and result rounded, 3 * 2^-24 at most where it counts) and by its additions, 32 in a block and nblocks / 256 + 11 behind
it; a probability also by its own argument's rounding, a log-probability by that of its size."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("V,n", [(1, 3), (3, 2), (31, 7), (1000, 5), (1023, 4), (1024, 9), (1025, 3), (2047, 2), (2048, 33), (2052, 3), (4097, 37),
                                 (10000, 160), (8191, 70), (70000, 2), (65569, 3), (10001, 3100), (10000, 3100), (100003, 40), (1000, 2000)])
def test_against_64_bits(ctx, V, n):
    r = np.random.default_rng(V + n)
    H = 16
    D = np.asfortranarray(r.uniform(-1, 1, (V, H)).astype(np.float32))
    b = r.uniform(-9, 3, V).astype(np.float32)
    h = np.asfortranarray(r.uniform(-1, 1, (H, n)).astype(np.float32))
    dD, db, dh = ctx.array(D), ctx.array(b), ctx.array(h)
    z, p, lp, at = ctx.empty((V, n)), ctx.empty((V, n)), ctx.empty((V, n)), ctx.array(np.full(V * n + 2, 7.0, np.float32))
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_PROB, p, z)
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_LOGPROB, lp, z)
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_PROB, at.at(1))  # in place, at an odd address
    ctx.sync()
    x = z.get().astype(np.float64)
    d = x - x.max(axis=0)
    want = d - np.log(np.exp(d).sum(axis=0))
    sums = (3 + 32 + V / 8192 + 11 + 4) * 2.0 ** -24
    assert np.all(np.abs(p.get() - np.exp(want)) <= np.exp(want) * (sums + np.abs(d) * 2.0 ** -24) + 2e-45)
    assert np.all(np.abs(lp.get() - want) <= sums + (np.abs(d) + 2 * np.abs(want) + 12) * 2.0 ** -24)
    got = at.get()
    assert got[0] == 7.0 and got[-1] == 7.0 and np.array_equal(got[1:-1].reshape((V, n), order="F"), p.get())


def test_infinite_logits(ctx):
    V, H, n = 3000, 16, 3
    b = np.zeros(V, np.float32)
    off = (np.arange(V) >= 2500) & (np.arange(V) % 32 != 5)  # (the product's own sum of a block of nothing but -inf is NaN)
    b[off] = -np.inf
    D, h = np.zeros((V, H), np.float32, order="F"), np.zeros((H, n), np.float32, order="F")
    dD, dh, p = ctx.array(D), ctx.array(h), ctx.empty((V, n))
    ctx.softmax_forward(dD, ctx.array(b), V, H, dh, n, capi.ZR_SOFTMAX_PROB, p)
    ctx.sync()
    assert np.all(p.get()[off] == 0.0) and np.allclose(p.get()[~off], 1.0 / np.sum(~off), rtol=1e-6)


def fold_of_one_large_logit(e, block):
    """The sum of 256 blocks, one a thread, in the kernels' order: 32 e each, but 1 in `block`."""
    p = np.full(256, np.float32(32) * np.float32(e), np.float32)
    p[block] = 1
    w, lanes = p.reshape(4, 64), np.arange(64)
    for off in (32, 16, 8, 4, 2, 1):
        w = w + w[:, lanes ^ off]
    return (w[0, 0] + w[1, 0]) + (w[2, 0] + w[3, 0])


@pytest.mark.parametrize("d", [9.732, 9.7779999, 10.41, 10.5, 10.782])
def test_blocks_far_below_one_large_logit(ctx, d):
    """The blocks' exponentials are those of expf, within one unit in the last place: exp2 of the rounded d * log2 e is off by 5 to 8 of them at
    these distances, all in the same direction."""
    V, H, block = 8192, 16, 77
    d = np.float32(d)
    b = np.zeros(V, np.float32)
    b[32 * block:32 * block + 32] = -1e30  # (nothing beside the one)
    b[32 * block + 3] = d
    out = ctx.empty((V + 2,))
    ctx.softmax_forward(ctx.zeros((V, H)), ctx.array(b), V, H, ctx.zeros((H, 1)), 1, capi.ZR_SOFTMAX_LOGITS, out)
    ctx.sync()
    mx, total = out.get()[V:]
    e = np.float32(np.exp(-np.float64(d)))
    assert mx == d
    assert fold_of_one_large_logit(np.nextafter(e, np.float32(0)), block) <= total <= fold_of_one_large_logit(np.nextafter(e, np.float32(1)), block)
