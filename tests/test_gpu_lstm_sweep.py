"""The whole sweep with streamed weights (csrc/zr_lstm_sweep.hip) against the oracle: sizes around the edges of its 32-row tiles, 32- and 64-column
tiles and steps of 64 k, columns off multiples of eight, infinities, and its rounding."""
import numpy as np
import pytest

import test_gpu_lstm_resident as r
from gpu_util import assert_close
from zoph_rnn_amd import capi, synth

pytestmark = pytest.mark.gpu

STREAMED = (capi.ZR_LSTM_STACK_PATH_SWEEP, capi.ZR_LSTM_SWEEP_STREAMED)


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    c.set_option(capi.ZR_OPT_LSTM_SWEEP, 2)
    yield c
    c.close()


# H: below a step, at and past one, an odd number of steps of 64 k, a row tile of 8; columns: one, past 8, 32 and 64, two and four
# tiles; layers whose 32-column tiles do not fit the chip take 64-column tiles
@pytest.mark.parametrize("H,mb,T,L", [(8, 1, 2, 1), (32, 9, 3, 3), (64, 33, 4, 2), (72, 7, 5, 2), (128, 65, 3, 4), (136, 100, 4, 2), (264, 31, 3, 8), (320, 129, 3, 4),
                                      (512, 250, 3, 4), (648, 37, 3, 2), (1000, 100, 3, 4), (1000, 63, 3, 4), (1032, 12, 2, 2)])
def test_sweep_with_streamed_weights(ctx, H, mb, T, L):
    c = r._case(H, mb, T, L)
    h, x, g, path, abandoned = r._run(ctx, c)
    h2, x2, g2, _, _ = r._run(ctx, c, times=3)
    assert path == STREAMED and not abandoned
    assert h.tobytes() == h2.tobytes() and x.tobytes() == x2.tobytes() and g.tobytes() == g2.tobytes()
    want_h, want_c = r._want(c)
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")
    m = (c["ids"] >= 0).astype(np.float32)[None, :, None, :]
    c_prev = np.concatenate([np.stack(c["c0"])[:, None], want_c[:, :-1]], axis=1)
    cell = np.clip(g[:, :, 1] * c_prev + g[:, :, 0] * g[:, :, 2], -0.9, 0.9)
    assert_close(m * cell, want_c, what="c from the gates")
    assert_close(m * g[:, :, 3] * np.tanh(cell), want_h, what="h from the gates")


# Terms of an infinite operand are infinity and NaN, and those of a value near the largest one may be: such sums are computed again.
@pytest.mark.parametrize("H,mb,L", [(8, 3, 1), (104, 8, 2), (320, 100, 1), (1000, 65, 4)])
def test_infinite_and_largest_inputs_saturate(ctx, H, mb, L):
    c = r._case(H, mb, 4, L)
    words = np.unique(c["ids"][c["ids"] >= 0])
    for i, v in enumerate(words):  # at most one such value a column: each gate's sum is then huge and saturates
        if i % 3:
            c["embed"][H - 1 - (i % min(H, 6)), v] = (np.inf, -np.inf, 3.4e38)[i % 3 if i % 2 else 1]
    c["h0"][0][H - 1, 0] = np.inf
    c["ids"][0, 0] = words[0]
    want_h, want_c = r._want(c)
    assert np.isfinite(want_h).all() and np.isfinite(want_c).all()
    h, x, _, path, _ = r._run(ctx, c)
    assert path == STREAMED
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")


@pytest.mark.parametrize("H,mb", [(64, 64), (256, 40), (512, 128), (1000, 200), (1024, 64)])
def test_rounds_no_more_than_one_launch_per_diagonal(ctx, H, mb):
    """The two schedules' errors against 64 bits, each an average over T * H * mb values, which vary by a few per cent between draws."""
    g, T, V = synth.rng(47, H + mb), 12, 300
    c = dict(H=H, mb=mb, T=T, L=1, V=V, ids=g.integers(0, V, size=(T, mb)).astype(np.int32), embed=synth.uniform(g, (H, V), -1, 1),
             layers=[r._rough_layer(g, H)], h0=[np.zeros((H, mb), np.float32)], c0=[np.zeros((H, mb), np.float32)])
    M, W, b = [r._wide(c["layers"][0], k) for k in ("M", "Wh", "b")]
    want, hp, cp = [], np.zeros((H, mb)), np.zeros((H, mb))
    for t in range(T):
        hp, cp = r._cell_in_64_bits(M @ c["embed"][:, c["ids"][t]].astype(np.float64) + W @ hp + b, cp)
        want.append(hp)
    error = {}
    for option in (1, 2):
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, option)
        try:
            h, _, _, path, _ = r._run(ctx, c, clip=0.0)
        finally:
            ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 2)
        assert (path == STREAMED) == (option == 2)
        error[option] = np.linalg.norm(h[0] - np.stack(want)) / np.linalg.norm(want)
    print(H, mb, error)
    assert error[2] < 1.1 * error[1]


def test_next_best_schedule_where_there_is_no_memory(ctx):
    """Estimated us of this size: streamed 305, resident 433, one launch per diagonal 516.  What a schedule may not have is not taken from the
    scratch buffer either, whose size the query tells."""
    H, mb, T, L = 704, 64, 12, 3
    c = r._case(H, mb, T, L)
    resident_kib = 4 * L * (T + 1) * H * mb // 1024 + 1  # the streamed sweep needs half as much again and the embedding columns
    want, paths, held = {}, {}, []
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 1)
    want["diagonals"] = r._run(ctx, c)[0]
    for option in (0, 2, 3):
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, option)
        for limit in (0, resident_kib, 1, 0):
            ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SCRATCH, limit)
            try:
                h, _, _, path, abandoned = r._run(ctx, c)
            finally:
                ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SCRATCH, 0)
            held.append(ctx.query(capi.ZR_QUERY_SCRATCH_KIB))
            assert not abandoned
            paths.setdefault((option, limit), []).append(path)
            assert np.array_equal(want.setdefault(path, h), h)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 2)
    diagonals = (capi.ZR_LSTM_STACK_PATH_DIAGONALS, 0)
    for option, first in ((0, STREAMED), (2, STREAMED), (3, r.RESIDENT)):
        assert paths[option, 0] == [first] * 2 and paths[option, resident_kib] == [r.RESIDENT] and paths[option, 1] == [diagonals], paths
    assert np.array_equal(want[diagonals], want["diagonals"])
    assert held == sorted(held), held
