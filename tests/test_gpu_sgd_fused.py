"""The clipped update in one launch whose workgroups exchange their sums (sgd_fused_kernel in csrc/zr_backward.hip): edges of its workgroups and of the
sizes that take two, four and eight accesses a thread, any alignment, waits that are given up, and launch numbers that start again.
Tolerance as in test_gpu_sgd_small.py; the same bits whether or not a wait was given up."""
import numpy as np
import pytest

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def check(ctx, n, off_w, off_g, clip, seed=0):
    r = np.random.default_rng(n + off_w + 8 * off_g + seed)
    w, g = r.uniform(-1, 1, n + 8).astype(np.float32), r.normal(0, 3, n + 8).astype(np.float32)
    dw, dg = ctx.array(w), ctx.array(g)
    scale, lr = 0.05, 0.7
    ctx.sgd_update(dw.at(off_w), dg.at(off_g), n, scale, clip, lr)
    ctx.sync()
    x = g[off_g:off_g + n].astype(np.float64) * np.float32(scale)
    step = np.float32(lr) * x * min(1.0, np.float32(clip) / np.linalg.norm(x))
    want = w.astype(np.float64)
    want[off_w:off_w + n] += step
    got = dw.get()
    assert np.array_equal(np.delete(got, np.s_[off_w:off_w + n]), np.delete(w, np.s_[off_w:off_w + n]))
    assert np.all(np.abs(got - want)[off_w:off_w + n] <= 2.0 ** -24 * (7 * np.abs(step) + np.abs(want[off_w:off_w + n])))


M = 1 << 20
SIZES = [28001, 32767, 32768, 32769, 65537, 250000, M - 1, M, M + 1, M + 3, 2 * M, 2 * M + 5, 4 * M - 2, 4 * M, 4 * M + 1]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off_w,off_g,clip", [(0, 0, 0.5), (1, 0, 0.5), (4, 3, 1e6)])
def test_update(ctx, n, off_w, off_g, clip):
    check(ctx, n, off_w, off_g, clip)


@pytest.mark.parametrize("n", [28001, 250000, 4 * M])
def test_a_workgroup_that_gives_up_forms_the_norm_itself(ctx, n):
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 1)
    try:
        check(ctx, n, 0, 0, 0.5)
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
    check(ctx, n, 0, 0, 0.5, 1)


def test_launch_numbers_start_again(ctx):
    check(ctx, 4 * M, 0, 0, 0.5)  # (slots that the next launches do not write)
    w, g = ctx.zeros((28001,)), ctx.zeros((28001,))
    for _ in range(65531):
        ctx.sgd_update(w, g, 28001, 1.0, 1.0, 0.1)
    for i in range(8):
        check(ctx, 4 * M if i % 2 else 28001, 0, 0, 0.5, i)


@pytest.mark.parametrize("special", [np.nan, np.inf])
def test_non_finite_gradients(ctx, special):
    n = 100000
    g = np.ones(n, np.float32)
    g[54321] = special
    dw = ctx.array(np.ones(n, np.float32))
    ctx.sgd_update(dw, ctx.array(g), n, 1.0, 5.0, 0.1)
    ctx.sync()
    # a norm that is no number is not above the threshold (the plain step); an infinite one makes every finite step zero, the infinite one NaN
    step = np.where(np.isnan(g), np.nan, np.float32(0.1)) if np.isnan(special) else np.where(np.isinf(g), np.nan, 0.0)
    assert np.array_equal(dw.get(), (np.float32(1) + step).astype(np.float32), equal_nan=True)


def test_the_sum_keeps_its_64_bits(ctx):
    """A gradient of two values whose norm lies just above the middle of two floats: the sum of squares with 37 bits would round the other way."""
    r = np.random.default_rng(5)
    x, y = (r.uniform(1, 2, 1 << 20).astype(np.float32) for _ in range(2))
    total = x.astype(np.float64) ** 2 + y.astype(np.float64) ** 2
    short = (total.view(np.uint64) & ~np.uint64(0xffff)).view(np.float64)
    norm = lambda s: np.sqrt(s).astype(np.float32)
    step = lambda s, v: (np.float32(1.0) / norm(s)) * v
    at = np.flatnonzero((step(total, x) != step(short, x)) | (step(total, y) != step(short, y)))
    assert len(at) >= 8
    for i in at[:8]:
        g = np.zeros(40000, np.float32)
        g[7], g[11] = x[i], y[i]
        w = ctx.zeros((40000,))
        ctx.sgd_update(w, ctx.array(g), 40000, 1.0, 1.0, 1.0)
        ctx.sync()
        got = w.get()
        assert (got[7], got[11]) == (step(total[i:i + 1], x[i])[0], step(total[i:i + 1], y[i])[0])


@pytest.mark.parametrize("n", [28001, 40000, 250001, M + 3, 4 * M])
def test_workgroups_that_gave_up_arrive_at_the_same_bits(ctx, n):
    r = np.random.default_rng(n)
    w, g = r.uniform(-1, 1, n).astype(np.float32), ctx.array(r.normal(0, 3, n).astype(np.float32))
    got = []
    for extra in (0, 3):  # (waits for a number that is never stored)
        ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, extra)
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 50 if extra else 0)
        try:
            dw = ctx.array(w)
            ctx.sgd_update(dw, g, n, 0.05, 0.5, 0.7)
            repaired = ctx.query(capi.ZR_QUERY_WAITS_REPAIRED)
            got.append(dw.get())
        finally:
            ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, 0)
            ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
        assert repaired == (capi.ZR_REPAIRED_SGD_UPDATE if extra else 0)
    assert np.array_equal(got[0], got[1])


def test_beside_another_context_two_launches(ctx):
    """No waits where another context's work may hold the compute units."""
    check(ctx, 250000, 0, 0, 0.5)
    ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, 3)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 50)
    other = capi.Context(0)
    try:
        check(ctx, 250000, 0, 0, 0.5)
        assert ctx.query(capi.ZR_QUERY_WAITS_REPAIRED) == 0
    finally:
        other.close()
        ctx.set_option(capi.ZR_OPT_LSTM_STEP_WAIT_EXTRA, 0)
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
