"""zr_lstm_node_backward with results that share memory: where the error of h_{t-1} is not wanted, the same buffer for both results (the error to
the layer below stays), and results over the gate errors, which nobody needs after an input's gradient."""
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


@pytest.mark.parametrize("H,mb", [(20, 3), (300, 37), (1000, 128)])
def test_results_that_overlap(ctx, H, mb):
    r = np.random.default_rng(H + mb)
    w = ctx.lstm_train_create([ctx.array(x) for x in weights(r, H)], [ctx.array(x) for x in weights(r, H)], H)
    f = lambda: ctx.array(np.asfortranarray(r.standard_normal((H, mb)).astype(np.float32)))  # noqa: E731
    gates = [ctx.array(np.asfortranarray(g)) for g in gate_values(r, H, mb)]
    c, cp, above, nxt, cnxt, mask = f(), f(), f(), f(), f(), ctx.array(np.ones(mb, np.int32))
    n = H * mb

    def run(h_prev, below, dgates):
        ctx.lstm_node_backward(w, mb, gates, c, cp, mask, above, nxt, cnxt, dgates, h_prev, ctx.empty((n,)), below)
        ctx.sync()
    block = ctx.empty((8 * n,))
    run(block.at(4 * n), block.at(6 * n), block)
    apart = block.get()
    d, h, b = apart[:4 * n], apart[4 * n:5 * n], apart[6 * n:7 * n]
    run(block.at(4 * n), None, block)
    h_only = block.get()[4 * n:5 * n]  # (one product alone may take other tiles than two)
    for _ in range(3):
        one = ctx.array(np.full(n, 7.0, np.float32))
        run(one, one, ctx.empty((4 * n,)))
        assert np.array_equal(one.get(), b)
        for at_h, at_b in ((0, 5 * n), (5 * n, 2 * n), (n, 2 * n), (4 * n + 8, 5 * n), (5 * n, 4 * n + 8), (n, None)):
            block = ctx.empty((8 * n,))
            run(block.at(at_h), None if at_b is None else block.at(at_b), block)
            want = apart.copy()
            want[:4 * n] = d
            want[at_h:at_h + n] = h if at_b is not None else h_only
            if at_b is not None:
                want[at_b:at_b + n] = b
            got, written = block.get(), np.zeros(8 * n, bool)
            written[:4 * n] = written[at_h:at_h + n] = True
            if at_b is not None:
                written[at_b:at_b + n] = True
            assert np.array_equal(got[written], want[written]), (at_h, at_b)
    ctx.lstm_train_destroy(w)
