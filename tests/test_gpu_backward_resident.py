"""The backward sweep with its weights in registers (csrc/zr_backward_resident.hip): tiles of 16 rows and columns with rows and columns left over,
each size class, one to nine layers in one launch and in several, with and without final errors, clamps and the error to the input, and the
repetition by one workgroup a column where a wait was abandoned.  Reference: the recurrence in 64 bits on the saved values.
Tolerance: that of the launches per diagonal (test_gpu_backward.py), whose products are the same fp32 sums of 4H terms."""
import numpy as np
import pytest

from gpu_util import assert_close
from test_gpu_backward_tiles import gate_values, weights
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def case(L, H, mb, T, tail):
    r = np.random.default_rng(H + 7 * mb + T)
    c = dict(M=[weights(r, H) for _ in range(L)], Wh=[weights(r, H) for _ in range(L)], gates=[[gate_values(r, H, mb) for _ in range(T)] for _ in range(L)],
             c=r.standard_normal((L, T, H, mb)).astype(np.float32), c0=r.standard_normal((L, H, mb)).astype(np.float32),
             top=r.standard_normal((T, H, mb)).astype(np.float32), mask=(r.random((T, mb)) > 0.15).astype(np.int32), hT=None, cT=None)
    if tail:
        c["hT"], c["cT"] = (r.standard_normal((L, H, mb)).astype(np.float32) for _ in range(2))
    return c


def reference(c, clip):
    L, T, H, mb = c["c"].shape
    clamp = (lambda x: np.clip(x, -clip, clip)) if clip else (lambda x: x)
    eh = [c["hT"][l].astype(np.float64) if c["hT"] is not None else np.zeros((H, mb)) for l in range(L)]
    ec = [c["cT"][l].astype(np.float64) if c["cT"] is not None else np.zeros((H, mb)) for l in range(L)]
    dg, below = np.zeros((L, T, 4 * H, mb)), np.zeros((T, H, mb))
    stacks = [[np.concatenate(c[k][l], axis=0).astype(np.float64) for k in ("Wh", "M")] for l in range(L)]
    for t in range(T - 1, -1, -1):
        above = c["top"][t].astype(np.float64)
        for l in range(L - 1, -1, -1):
            e = ((above if l == L - 1 else clamp(above)) + clamp(eh[l])) * c["mask"][t]
            i, f, g, o = c["gates"][l][t].astype(np.float64)
            th = np.tanh(c["c"][l, t].astype(np.float64))
            x = (ec[l] + e * o * (1 - th * th)) * c["mask"][t]
            before = c["c"][l, t - 1] if t else c["c0"][l]
            dg[l, t] = np.concatenate([x * g * i * (1 - i), x * before * f * (1 - f), x * i * (1 - g * g), e * th * o * (1 - o)])
            ec[l] = x * f
            eh[l], above = stacks[l][0].T @ dg[l, t], stacks[l][1].T @ dg[l, t]
        below[t] = above
    return dg, below, [clamp(e) for e in eh], ec


def run(ctx, c, clip, want_below, option):
    L, T, H, mb = c["c"].shape
    flat = lambda x: ctx.array(np.ascontiguousarray(np.swapaxes(x, -1, -2), np.float32).reshape(-1))
    layers = [ctx.lstm_train_create([ctx.array(w) for w in c["M"][l]], [ctx.array(w) for w in c["Wh"][l]], H) for l in range(L)]
    each = lambda x: None if x is None else [flat(x[l]) for l in range(L)]
    dg = [ctx.empty((T * mb * 4 * H,)) for _ in range(L)]
    eh, ec, ein = [ctx.empty((H, mb)) for _ in range(L)], [ctx.empty((H, mb)) for _ in range(L)], ctx.empty((T * mb * H,))
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, option)
    try:
        for _ in range(2):  # the second time the flags are what the first left
            ctx.lstm_stack_backward(layers, T, mb, ctx.array(c["mask"].reshape(-1)), each(c["c0"]), each(c["c"]), [flat(np.stack(g)) for g in c["gates"]],
                                    flat(c["top"]), dg, eh, ec, err_hT=each(c["hT"]), err_cT=each(c["cT"]), d_err_below0=ein if want_below else None,
                                    err_clip=clip)
        ctx.sync()
        if option >= 2:
            assert ctx.query(capi.ZR_QUERY_LSTM_BACKWARD_PATH) == capi.ZR_LSTM_BACKWARD_PATH_RESIDENT
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 0)
        for w in layers:
            ctx.lstm_train_destroy(w)
    return ([x.get().reshape(T, mb, 4 * H).transpose(0, 2, 1) for x in dg], ein.get().reshape(T, mb, H).transpose(0, 2, 1) if want_below else None,
            [x.get() for x in eh], [x.get() for x in ec])


def compare(got, want):
    for l in range(len(got[0])):
        assert_close(got[0][l], want[0][l], what="gate errors, layer %d" % l)
        assert_close(got[2][l], want[2][l], what="error to h_0, layer %d" % l)
        assert_close(got[3][l], want[3][l], what="error to c_0, layer %d" % l)
    if got[1] is not None:
        assert_close(got[1], want[1], what="error to the input")


SIZES = [(1, 8, 1, 1), (1, 8, 3, 5), (2, 20, 17, 4), (3, 100, 20, 7), (2, 128, 16, 3), (4, 129, 33, 5), (2, 256, 15, 4), (2, 300, 20, 6), (1, 321, 40, 3),
         (2, 384, 16, 3), (2, 385, 24, 3), (2, 500, 64, 4), (1, 512, 100, 3), (5, 500, 50, 3), (9, 64, 16, 3), (4, 320, 48, 12)]


@pytest.mark.parametrize("L,H,mb,T", SIZES)
@pytest.mark.parametrize("tail,clip,below", [(False, 0.0, True), (True, 0.1, True), (True, 0.0, False)])
def test_sweep(ctx, L, H, mb, T, tail, clip, below):
    c = case(L, H, mb, T, tail)
    want = reference(c, clip)
    compare(run(ctx, c, clip, below, 3), want)


@pytest.mark.parametrize("L,H,mb,T", [(1, 8, 3, 5), (3, 100, 20, 7), (2, 500, 64, 4), (5, 500, 50, 3)])
def test_an_abandoned_sweep_is_formed_again(ctx, L, H, mb, T):
    """With one poll a wait workgroups give up; the results are right all the same and nothing is reported."""
    c = case(L, H, mb, T, True)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 1)
    try:
        got = run(ctx, c, 0.1, True, 3)
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
    compare(got, reference(c, 0.1))
    compare(run(ctx, c, 0.1, True, 3), reference(c, 0.1))


@pytest.mark.parametrize("L,H,mb,T", [(1, 8, 1, 1), (1, 8, 3, 5), (3, 100, 20, 7), (2, 385, 24, 3), (5, 500, 50, 3), (9, 64, 16, 3)])
@pytest.mark.parametrize("clip,below", [(0.1, True), (0.0, False)])
def test_waits_that_cannot_end_are_given_up_and_the_sweep_formed_again(ctx, L, H, mb, T, clip, below):
    """Every wait expects more slots than there are: each launch is abandoned, whatever the timing."""
    c = case(L, H, mb, T, True)
    ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, 1)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 30)
    try:
        got = run(ctx, c, clip, below, 3)
        repaired = ctx.query(capi.ZR_QUERY_WAITS_REPAIRED)
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, 0)
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
    assert repaired & capi.ZR_REPAIRED_LSTM_BACKWARD
    compare(got, reference(c, clip))
    compare(run(ctx, c, clip, below, 3), reference(c, clip))
    assert ctx.query(capi.ZR_QUERY_WAITS_REPAIRED) & capi.ZR_REPAIRED_LSTM_BACKWARD == 0


def test_results_on_operands_take_the_launches_per_diagonal(ctx):
    """err_below0 written over err_top, err_c0 over err_cT: as before the single launch."""
    L, H, mb, T = 2, 64, 8, 4
    c = case(L, H, mb, T, True)
    flat = lambda x: ctx.array(np.ascontiguousarray(np.swapaxes(x, -1, -2), np.float32).reshape(-1))
    layers = [ctx.lstm_train_create([ctx.array(w) for w in c["M"][l]], [ctx.array(w) for w in c["Wh"][l]], H) for l in range(L)]
    top, cT = flat(c["top"]), [flat(c["cT"][l]) for l in range(L)]
    dg, eh = [ctx.empty((T * mb * 4 * H,)) for _ in range(L)], [ctx.empty((H, mb)) for _ in range(L)]
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 1)  # (would show an operand read again)
    try:
        ctx.lstm_stack_backward(layers, T, mb, ctx.array(c["mask"].reshape(-1)), [flat(x) for x in c["c0"]], [flat(x) for x in c["c"]],
                                [flat(np.stack(g)) for g in c["gates"]], top, dg, eh, cT, err_hT=[flat(x) for x in c["hT"]], err_cT=cT, d_err_below0=top)
        ctx.sync()
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
    assert ctx.query(capi.ZR_QUERY_LSTM_BACKWARD_PATH) == capi.ZR_LSTM_BACKWARD_PATH_DIAGONALS
    want = reference(c, 0.0)
    by_column = lambda a, *s: a.get().reshape(*s).swapaxes(-1, -2)
    compare(([by_column(x, T, mb, 4 * H) for x in dg], by_column(top, T, mb, H), [x.get() for x in eh], [by_column(x, mb, H) for x in cT]), want)
    for w in layers:
        ctx.lstm_train_destroy(w)


def test_results_on_one_another_are_written_in_the_diagonals_order(ctx):
    """One array for the error to every layer's initial h: the last layer's stays."""
    L, H, mb, T = 3, 64, 8, 4
    c = case(L, H, mb, T, True)
    flat = lambda x: ctx.array(np.ascontiguousarray(np.swapaxes(x, -1, -2), np.float32).reshape(-1))
    layers = [ctx.lstm_train_create([ctx.array(w) for w in c["M"][l]], [ctx.array(w) for w in c["Wh"][l]], H) for l in range(L)]
    dg, ec, eh = [ctx.empty((T * mb * 4 * H,)) for _ in range(L)], [ctx.empty((H, mb)) for _ in range(L)], ctx.empty((H, mb))
    ctx.lstm_stack_backward(layers, T, mb, ctx.array(c["mask"].reshape(-1)), [flat(x) for x in c["c0"]], [flat(x) for x in c["c"]],
                            [flat(np.stack(g)) for g in c["gates"]], flat(c["top"]), dg, [eh] * L, ec, err_hT=[flat(x) for x in c["hT"]],
                            err_cT=[flat(x) for x in c["cT"]])
    ctx.sync()
    assert ctx.query(capi.ZR_QUERY_LSTM_BACKWARD_PATH) == capi.ZR_LSTM_BACKWARD_PATH_DIAGONALS
    want = reference(c, 0.0)
    assert_close(eh.get(), want[2][L - 1], what="error to h_0 of the last layer")
    for l in range(L):
        assert_close(ec[l].get(), want[3][l], what="error to c_0, layer %d" % l)
    for w in layers:
        ctx.lstm_train_destroy(w)


def test_without_an_option_the_same_sizes_take_one_launch(ctx):
    """(what the two tests before this one would take if no memory were shared)"""
    for L, H, mb, T in ((2, 64, 8, 4), (3, 64, 8, 4)):
        c = case(L, H, mb, T, True)
        compare(run(ctx, c, 0.0, True, 0), reference(c, 0.0))
        assert ctx.query(capi.ZR_QUERY_LSTM_BACKWARD_PATH) == capi.ZR_LSTM_BACKWARD_PATH_RESIDENT
