"""The error products of the backward pass, W_h^T dg and M^T dg, over the tiles they can run on: 32 x 32 with K split over
eight waves, up to 256 of them a grouped launch (two nodes of H = 1000 at 64 columns) or, beyond 32 columns, 384 (the same at
65 columns), 64 x 64 beyond, and hidden sizes that are no multiple of four.  Each is compared with the product in 64 bits of the
gate errors the library itself left.
Tolerance: K = 4H products and their sums, each rounded to fp32 at most once a term: (4H + 2) 2^-24 of the sum of the terms'
magnitudes."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu

SIZES = [(127, 3), (128, 1), (130, 33), (132, 20), (160, 32), (300, 65), (500, 64), (1000, 16), (1000, 64), (1000, 65), (1000, 128)]


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def check(got, W, dg):
    """got (H x mb) against sum_g W[g]^T dg_g, dg (4H x mb)."""
    stack = np.concatenate(W, axis=0).astype(np.float64)
    d = dg.astype(np.float64)
    assert np.all(np.abs(got - stack.T @ d) <= (stack.shape[0] + 2) * 2.0 ** -24 * (np.abs(stack).T @ np.abs(d)))


def weights(r, H):
    return [np.asfortranarray(r.uniform(-0.08, 0.08, (H, H)).astype(np.float32)) for _ in range(4)]


def gate_values(r, H, mb):
    g = r.uniform(0.05, 0.95, (4, H, mb)).astype(np.float32)
    g[2] = 2 * g[2] - 1
    return g


@pytest.mark.parametrize("H,mb", SIZES)
def test_two_nodes_of_a_diagonal(ctx, H, mb):
    r = np.random.default_rng(H + 7 * mb)
    L = T = 2
    M, Wh = [weights(r, H) for _ in range(L)], [weights(r, H) for _ in range(L)]
    layers = [ctx.lstm_train_create([ctx.array(w) for w in M[l]], [ctx.array(w) for w in Wh[l]], H) for l in range(L)]
    flat = lambda x: ctx.array(np.ascontiguousarray(x, np.float32).reshape(-1))
    by_column = lambda x: np.swapaxes(x, -1, -2)  # host (.., H, mb) -> device order (.., mb, H)
    mask = ctx.array(np.ones(T * mb, np.int32))
    gates = [flat(np.stack([by_column(gate_values(r, H, mb)) for _ in range(T)])) for _ in range(L)]
    c = [flat(r.standard_normal((T, mb, H))) for _ in range(L)]
    c0, top = flat(r.standard_normal((mb, H))), flat(r.standard_normal((T, mb, H)))
    dg = [ctx.empty((T * mb * 4 * H,)) for _ in range(L)]
    eh, ec, ein = [ctx.empty((H, mb)) for _ in range(L)], [ctx.empty((H, mb)) for _ in range(L)], ctx.empty((T * mb * H,))
    ctx.lstm_stack_backward(layers, T, mb, mask, [c0] * L, c, gates, top, dg, eh, ec, d_err_below0=ein)
    ctx.sync()
    d = [x.get().reshape(T, mb, 4 * H).transpose(0, 2, 1) for x in dg]
    below = ein.get().reshape(T, mb, H).transpose(0, 2, 1)
    for l in range(L):
        check(eh[l].get(), Wh[l], d[l][0])
    for t in range(T):
        check(below[t], M[0], d[0][t])
    for w in layers:
        ctx.lstm_train_destroy(w)


@pytest.mark.parametrize("H,mb", SIZES)
@pytest.mark.parametrize("adjacent", [True, False])
def test_one_node(ctx, H, mb, adjacent):
    r = np.random.default_rng(H + 11 * mb)
    M, Wh = weights(r, H), weights(r, H)
    layer = ctx.lstm_train_create([ctx.array(w) for w in M], [ctx.array(w) for w in Wh], H)
    column = lambda: ctx.array(np.asfortranarray(r.standard_normal((H, mb)).astype(np.float32)))
    gates = [ctx.array(np.asfortranarray(g)) for g in gate_values(r, H, mb)]
    dg, out, other = ctx.empty((4 * H, mb)), ctx.empty((H, 2 * mb)), ctx.empty((H, mb))
    below = int(out.ptr) + 4 * H * mb if adjacent else other
    ctx.lstm_node_backward(layer, mb, gates, column(), column(), ctx.array(np.ones(mb, np.int32)), column(), None, None, dg, out,
                           ctx.empty((H, mb)), below)
    ctx.sync()
    d, o = dg.get(), out.get()
    check(o[:, :mb], Wh, d)
    check(o[:, mb:] if adjacent else other.get(), M, d)
    ctx.lstm_train_destroy(layer)
