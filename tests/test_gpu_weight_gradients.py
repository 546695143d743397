"""Weight and bias gradients of a layer in one launch (csrc/zr_weight_gradients.hip): rows and columns left over in its 64 x 64 tiles, fewer columns than a
wave takes at a time, one step (no array of later states), and gradients added to what is there.
Tolerance: N products and their sums, each rounded to fp32 at most once a term, a dozen sums behind them: (N + 14) 2^-24 of the sum of the terms'
magnitudes, and one rounding of the result."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def operands(H, T, mb):
    r = np.random.default_rng(H + 100 * T + mb)
    n = T * mb
    return [r.standard_normal(s).astype(np.float32) for s in ((n, 4 * H), (n, H), (mb, H), (n, H))]


def check(got, a, b, before=0.0):
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = (a.T @ b).T + before
    bound = (a.shape[0] + 14) * 2.0 ** -24 * (np.abs(a).T @ np.abs(b)).T + 2.0 ** -23 * np.abs(want)
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("H,T,mb", [(1, 1, 1), (2, 3, 5), (8, 1, 130), (15, 2, 8), (16, 9, 7), (17, 16, 8), (33, 5, 13), (63, 4, 33), (65, 3, 50), (100, 20, 20), (129, 8, 16),
                                    (300, 35, 20), (333, 7, 33), (500, 24, 64), (501, 1, 64), (700, 5, 64)])
def test_gradients(ctx, H, T, mb):
    dg, x, h0, h = operands(H, T, mb)
    flat = lambda v: ctx.array(v.reshape(-1))
    dM, dWh, db = ctx.empty((H, 4 * H)), ctx.empty((H, 4 * H)), ctx.empty((4 * H,))
    ctx.lstm_weight_gradients(H, T, mb, flat(dg), flat(x), flat(h0), flat(h) if T > 1 else None, dM, dWh, db)
    ctx.sync()
    as_rows = lambda d: d.get().reshape(-1, order="F").reshape(H, 4 * H)
    check(as_rows(dM), dg, x)
    check(as_rows(dWh), dg, np.concatenate([h0, h[:(T - 1) * mb]]))
    check(db.get()[None, :], dg, np.ones((T * mb, 1), np.float32))


@pytest.mark.parametrize("H,mb", [(5, 3), (64, 16), (100, 70), (500, 64)])
def test_gradients_of_one_node_are_added(ctx, H, mb):
    dg, x, h0, _ = operands(H, 1, mb)
    flat = lambda v: ctx.array(v.reshape(-1))
    r = np.random.default_rng(9)
    old = [r.standard_normal(4 * H * H).astype(np.float32), r.standard_normal(4 * H * H).astype(np.float32), r.standard_normal(4 * H).astype(np.float32)]
    out = [ctx.array(o) for o in old]
    ctx.lstm_node_gradients(H, mb, flat(dg), flat(x), flat(h0), *out)
    ctx.sync()
    check(out[0].get().reshape(H, 4 * H), dg, x, old[0].reshape(H, 4 * H).astype(np.float64))
    check(out[1].get().reshape(H, 4 * H), dg, h0, old[1].reshape(H, 4 * H).astype(np.float64))
    check(out[2].get()[None, :], dg, np.ones((mb, 1), np.float32), old[2][None, :].astype(np.float64))


@pytest.mark.parametrize("H,T,mb", [(33, 5, 13), (100, 20, 20)])
def test_results_that_share_memory_are_formed_one_after_another(ctx, H, T, mb):
    dg, x, h0, h = operands(H, T, mb)
    flat = lambda v: ctx.array(v.reshape(-1))
    prev = np.concatenate([h0, h[:(T - 1) * mb]])
    as_rows = lambda d: d.get().reshape(-1, order="F").reshape(H, 4 * H)
    dM, dWh, db = ctx.empty((H, 4 * H)), ctx.empty((H, 4 * H)), ctx.empty((4 * H,))
    ctx.lstm_weight_gradients(H, T, mb, flat(dg), flat(x), flat(h0), flat(h), dM, dM, db)  # the later one stays
    ctx.sync()
    check(as_rows(dM), dg, prev)
    # over the columns that only it reads
    n = max(T * mb * H, 4 * H * H)
    x_and_dM = ctx.array(np.concatenate([x.reshape(-1), np.zeros(n - T * mb * H, np.float32)]))
    ctx.lstm_weight_gradients(H, T, mb, flat(dg), x_and_dM, flat(h0), flat(h), x_and_dM, dWh, db)
    ctx.sync()
    check(x_and_dM.get()[:4 * H * H].reshape(H, 4 * H), dg, x)
    check(as_rows(dWh), dg, prev)
    check(db.get()[None, :], dg, np.ones((T * mb, 1), np.float32))


@pytest.mark.parametrize("H,mb", [(5, 3), (64, 16), (100, 70)])
def test_gradients_of_one_node_added_into_one_array(ctx, H, mb):
    dg, x, h0, _ = operands(H, 1, mb)
    flat = lambda v: ctx.array(v.reshape(-1))
    dW, db = ctx.zeros((4 * H * H,)), ctx.zeros((4 * H,))
    ctx.lstm_node_gradients(H, mb, flat(dg), flat(x), flat(h0), dW, dW, db)
    ctx.sync()
    check(dW.get().reshape(H, 4 * H), np.concatenate([dg, dg]), np.concatenate([x, h0]))
    check(db.get()[None, :], dg, np.ones((mb, 1), np.float32))
