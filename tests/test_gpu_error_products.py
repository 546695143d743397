"""The error products of a full diagonal on the bf16 matrix cores (csrc/zr_error_products.hip): K around the revolutions of the operand ring, 64 x 64
tiles with rows and columns left over, one to nine layers, and gate errors that are infinite.
Tolerance: six exact products a pair of values, each added with at most one rounding to fp32, so K = 4H additions of six products and two dozen
sums: (4H + 24) 2^-24 of the sum of the terms' magnitudes; the terms left out are below one more."""
import numpy as np
import pytest

from test_gpu_backward_tiles import gate_values, weights
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def run(ctx, L, H, mb, top):
    r = np.random.default_rng(H + 7 * mb)
    T = L
    M, Wh = [weights(r, H) for _ in range(L)], [weights(r, H) for _ in range(L)]
    layers = [ctx.lstm_train_create([ctx.array(w) for w in M[l]], [ctx.array(w) for w in Wh[l]], H) for l in range(L)]
    flat = lambda x: ctx.array(np.ascontiguousarray(x, np.float32).reshape(-1))
    by_column = lambda x: np.swapaxes(x, -1, -2)
    mask = ctx.array(np.ones(T * mb, np.int32))
    gates = [flat(np.stack([by_column(gate_values(r, H, mb)) for _ in range(T)])) for _ in range(L)]
    c = [flat(r.standard_normal((T, mb, H))) for _ in range(L)]
    c0 = flat(r.standard_normal((mb, H)))
    dg = [ctx.empty((T * mb * 4 * H,)) for _ in range(L)]
    eh, ec, ein = [ctx.empty((H, mb)) for _ in range(L)], [ctx.empty((H, mb)) for _ in range(L)], ctx.empty((T * mb * H,))
    ctx.lstm_stack_backward(layers, T, mb, mask, [c0] * L, c, gates, flat(top(r, T)), dg, eh, ec, d_err_below0=ein)
    ctx.sync()
    for w in layers:
        ctx.lstm_train_destroy(w)
    return M, Wh, [x.get().reshape(T, mb, 4 * H).transpose(0, 2, 1) for x in dg], [x.get() for x in eh], ein.get().reshape(T, mb, H).transpose(0, 2, 1)


# the diagonal of all layers has more than 256 tiles of 32 x 32; hidden sizes even, every remainder of 64 rows' halves
@pytest.mark.parametrize("L,H,mb", [(4, 100, 300), (9, 132, 129), (4, 260, 130), (3, 300, 192), (2, 516, 193), (4, 500, 65), (1, 1028, 128), (2, 1000, 160)])
def test_against_64_bits(ctx, L, H, mb):
    M, Wh, d, eh, below = run(ctx, L, H, mb, lambda r, T: r.standard_normal((T, mb, H)))
    pairs = [(eh[l], Wh[l], d[l][0]) for l in range(L)] + [(below[t], M[0], d[0][t]) for t in range(L)]
    for got, W, dg in pairs:
        stack, x = np.concatenate(W, axis=0).astype(np.float64), dg.astype(np.float64)
        assert np.all(np.abs(got - stack.T @ x) <= (4 * H + 25) * 2.0 ** -24 * (np.abs(stack).T @ np.abs(x)))


def test_infinite_errors_stay_in_their_columns(ctx):
    L, H, mb = 1, 1000, 256

    def top(r, T):
        x = r.standard_normal((T, mb, H))
        x[0, 77, 5], x[0, 200, 999] = np.inf, 3e38
        return x
    M, Wh, d, eh, below = run(ctx, L, H, mb, top)
    for got, W in ((eh[0], Wh[0]), (below[0], M[0])):
        with np.errstate(all="ignore"):
            want = np.concatenate(W, axis=0).astype(np.float64).T @ d[0][0].astype(np.float64)
        finite = np.isfinite(d[0][0]).all(0)
        assert not finite[77] and finite[[76, 78]].all()
        assert not np.isfinite(got[:, 77]).any()
        fine = finite & (np.abs(want).max(0) < 3e38)
        assert fine.sum() >= mb - 2
        scale = np.abs(np.concatenate(W, axis=0).astype(np.float64)).T @ np.abs(d[0][0][:, fine].astype(np.float64))
        assert np.all(np.abs(got[:, fine] - want[:, fine]) <= (4 * H + 25) * 2.0 ** -24 * scale)
