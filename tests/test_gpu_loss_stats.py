"""The 64-bit column statistics behind zr_softmax_loss and zr_softmax_logprob_f64 (csrc/zr_softmax.hip): columns shorter than a load,
a round of loads and its edges, columns shared by several workgroups, unaligned columns, infinite and NaN logits.  The
reference is taken from the very logits the call leaves in its scratch matrix, so only the 64-bit sums differ: V
additions of non-negative terms and one exp of an argument rounded once, below (V + 8) * 2^-52 of the sum, hence of the
logarithm in absolute terms."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def run(ctx, V, n, special=None):
    r = np.random.default_rng(V + 7 * n)
    H = 24
    D = np.asfortranarray(r.uniform(-0.5, 0.5, (V, H)).astype(np.float32))
    b = r.uniform(-4, 4, V).astype(np.float32)
    if special is not None:
        b[V // 2:] = special
    h = np.asfortranarray(r.uniform(-1, 1, (H, n)).astype(np.float32))
    target = r.integers(0, max(1, V // 2), n).astype(np.int32)
    mask = (np.arange(n) % 3 != 1).astype(np.int32)
    dD, db, dh = ctx.array(D), ctx.array(b), ctx.array(h)
    x, lp = ctx.empty((V, n)), ctx.empty((V, n), np.float64)
    loss = ctx.softmax_loss(dD, db, V, H, dh, n, ctx.array(target), ctx.array(mask), x)
    z = x.get().astype(np.float64)
    ctx.softmax_logprob_f64(dD, db, V, H, dh, n, lp, x)
    ctx.sync()
    assert np.array_equal(x.get().astype(np.float64), z, equal_nan=True)
    return z, loss, lp.get(), target, mask


@pytest.mark.parametrize("V,n", [(1, 1), (3, 2), (4, 700), (31, 5), (2047, 3), (8191, 1), (8192, 2), (8195, 3), (16390, 1), (33333, 1), (33333, 70),
                                 (50000, 12), (12289, 513), (10001, 600)])
def test_against_64_bits(ctx, V, n):
    z, loss, lp, target, mask = run(ctx, V, n)
    m = z.max(axis=0)
    want = (z - m) - np.log(np.exp(z - m).sum(axis=0))
    bound = (V + 8) * 2.0 ** -52
    assert np.all(np.abs(lp - want) <= bound + 2.0 ** -52 * np.abs(want))
    per = want[target, np.arange(n)] * mask
    assert abs(loss - per.sum()) <= n * bound + (n + 2) * 2.0 ** -52 * np.abs(per).sum()


def test_infinite_and_nan_logits(ctx):
    z, loss, lp, target, mask = run(ctx, 8300, 3, -np.inf)  # the lower half has probability 0
    k = 4150
    m = z[:k].max(axis=0)
    want = (z[:k] - m) - np.log(np.exp(z[:k] - m).sum(axis=0))
    assert np.all(np.abs(lp[:k] - want) <= (k + 8) * 2.0 ** -52 + 2.0 ** -52 * np.abs(want))
    assert np.all(lp[k:] == -np.inf) and np.isfinite(loss)
    for special in (np.inf, np.nan):
        _, loss, lp, _, _ = run(ctx, 8300, 3, special)
        assert np.isnan(loss) and np.all(np.isnan(lp[:k]))
