"""The attention node's backward pass where the error of h_t is written over c_t, or weight gradients share their memory: the same bits as with memory of
their own, whether the four weight gradients are one launch (up to 256 columns) or products one after another."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


KEYS = ("W_a", "W_p", "v_p", "bias", "W_c1", "W_c2")


class Node:
    def __init__(self, ctx, H, mb, S=5, D=2):
        self.ctx, self.H, self.mb, self.S = ctx, H, mb, S
        r = np.random.default_rng(H + mb)
        U = lambda *s: ctx.array(r.uniform(-0.3, 0.3, s).astype(np.float32))
        self.keep = tables, dw = [U(H, mb) for _ in range(S)], {k: U(H) if k in ("v_p", "out_bias") else U(H, H) for k in ("W_a", "W_p", "v_p", "out_bias", "W_c1", "W_c2")}
        self.a = ctx.attn_create(H, mb, D, dw["W_a"], dw["W_p"], dw["v_p"], dw["out_bias"], dw["W_c1"], dw["W_c2"], tables)
        self.errors = [ctx.zeros((H, mb)) for _ in range(S)]
        ctx.attn_set_error_tables(self.a, self.errors)
        lens = r.integers(1, S + 1, mb).astype(np.int32)
        self.info, self.h, self.mask = ctx.array(np.concatenate([lens, S - lens]).astype(np.int32)), U(H, mb), ctx.array((r.random(mb) > 0.1).astype(np.int32))
        W = 2 * D + 1
        self.htild, self.align, self.index, self.p, self.c = (ctx.empty((H, mb)), ctx.empty((mb, W)), ctx.empty((mb, W), np.int32), ctx.empty((mb,)),
                                                              ctx.empty((H, mb)))
        ctx.attn_step(self.a, self.info, self.h, self.mask, self.htild, self.align, self.index, self.p, self.c)
        self.err = U(H, mb)

    def backward(self, shared=(), on_c=False):
        """`shared`: names of weight gradients that are one array.  Returns (error of h_t, gradients by name)."""
        ctx, H, mb = self.ctx, self.H, self.mb
        for e in self.errors:
            e.set(np.zeros((H, mb), np.float32))
        one = ctx.zeros((H, H))
        g = {k: one if k in shared else ctx.zeros((H,) if k in ("v_p", "bias") else (H, H)) for k in KEYS}
        out, c = ctx.empty((H, mb)), ctx.array(self.c.get())
        ctx.attn_backward(self.a, self.info, self.h, self.mask, self.htild, self.align, self.index, self.p, c, self.err, c if on_c else out, [g[k] for k in KEYS])
        ctx.sync()
        return (c if on_c else out).get(), {k: v.get() for k, v in g.items()}


SIZES = [(33, 7), (64, 64), (100, 256), (100, 257)]


@pytest.mark.parametrize("H,mb", SIZES)
def test_error_over_the_context(ctx, H, mb):
    node = Node(ctx, H, mb)
    want_e, want = node.backward()
    got_e, got = node.backward(on_c=True)
    assert np.array_equal(got_e, want_e)
    for k in KEYS:
        assert np.array_equal(got[k], want[k]), k
    ctx.attn_destroy(node.a)


@pytest.mark.parametrize("H,mb", SIZES)
@pytest.mark.parametrize("shared", [("W_c1", "W_p"), ("W_c2", "W_a"), ("W_c1", "W_c2"), ("W_p", "W_a"), ("W_c1", "W_c2", "W_p", "W_a")])
def test_gradients_added_into_one_array(ctx, H, mb, shared):
    node = Node(ctx, H, mb)
    want_e, want = node.backward()
    got_e, got = node.backward(shared)
    sums = np.zeros((H, H), np.float32)
    for k in ("W_c1", "W_c2", "W_p", "W_a"):  # one after another, in the order of the node's equations
        if k in shared:
            sums += want[k]
    assert np.array_equal(got_e, want_e)
    for k in KEYS:
        assert np.array_equal(got[k], sums if k in shared else want[k]), k
    ctx.attn_destroy(node.a)
