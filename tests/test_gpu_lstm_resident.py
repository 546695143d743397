"""The LSTM kernels on narrow row tiles: the whole sweep with weights in registers (zr_lstm_resident.hip) and one node
(zr_lstm_rows.hip), against the oracle: hidden
sizes around the edges of its row tiles, k-groups and register classes, batches around the edges of its column tiles,
more layers than fit in one launch, initial states, padding, cell clipping, kept gates, and giving up a wait."""
import numpy as np
import pytest

import oracle_lib as o
from gpu_util import Layer, assert_close
from zoph_rnn_amd import capi, synth

pytestmark = pytest.mark.gpu

RESIDENT = (capi.ZR_LSTM_STACK_PATH_SWEEP, capi.ZR_LSTM_SWEEP_RESIDENT)


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def _case(H, mb, T, L, V=211, seed=41):
    g = synth.rng(seed, H + 31 * mb + L)
    ids = g.integers(0, V, size=(T, mb)).astype(np.int32)
    if mb > 1:
        ids[: T // 2, 1] = -1
    ids[T - 1, mb - 1] = -1
    return dict(H=H, mb=mb, T=T, L=L, V=V, ids=ids, embed=synth.uniform(g, (H, V), -0.5, 0.5),
                layers=[synth.lstm_layer(g, H, forget_bias_one=True) for _ in range(L)],
                h0=[np.tanh(synth.uniform(g, (H, mb), -1, 1)) for _ in range(L)],
                c0=[synth.uniform(g, (H, mb), -0.5, 0.5) for _ in range(L)])


def _run(ctx, c, clip=0.9, times=1):
    """h, c and gates of every node, [L][T](, 4), H x mb."""
    H, mb, T, L, V, ids = c["H"], c["mb"], c["T"], c["L"], c["V"], c["ids"]
    layers = [Layer(ctx, ly) for ly in c["layers"]]
    d_nn, d_m = ctx.empty(ids.size, np.int32), ctx.empty(ids.size, np.int32)
    ctx.vocab_prep(ctx.array(ids.reshape(-1)), ids.size, V, d_nn, d_m)
    d_embed = ctx.array(c["embed"])
    d_h0, d_c0 = [ctx.array(a) for a in c["h0"]], [ctx.array(a) for a in c["c0"]]
    n = H * mb
    h, x = [ctx.empty((n * T,)) for _ in range(L)], [ctx.empty((n * T,)) for _ in range(L)]
    g = [ctx.empty((4 * n * T,)) for _ in range(L)]
    try:
        for _ in range(times):
            ctx.lstm_stack_forward_train([ly.w for ly in layers], d_embed, V, d_nn, d_m, T, mb, d_h0, d_c0, h, x, g, clip=clip)
        path = (ctx.query(capi.ZR_QUERY_LSTM_STACK_PATH), ctx.query(capi.ZR_QUERY_LSTM_SWEEP_KERNEL))
        abandoned = ctx.query(capi.ZR_QUERY_LSTM_SWEEP_ABANDONED)
    finally:
        for ly in layers:
            ly.close()
    shape = lambda a, k: a.get().reshape(T, *k, mb, H).swapaxes(-1, -2)  # noqa: E731
    return np.stack([shape(a, ()) for a in h]), np.stack([shape(a, ()) for a in x]), np.stack([shape(a, (4,)) for a in g]), path, abandoned


def _want(c, clip=0.9):
    nn, m = o.vocab_prep(c["ids"])
    return o.lstm_stack_forward(c["embed"], c["layers"], nn, m, h0=c["h0"], c0=c["c0"], clip=clip)


# H: one row tile, a row tail of every kind (H % 8 = 1, 4, 7), the last and first size of each register class;
# mb: 1, the last and first of 16 and 32 columns, several column tiles; L: one, several, more than fit at once
@pytest.mark.parametrize("H,mb,T,L", [(8, 1, 1, 1), (9, 16, 4, 2), (15, 17, 3, 3), (100, 8, 6, 1), (127, 33, 4, 2),
                                      (129, 5, 3, 8), (255, 32, 3, 2), (257, 31, 3, 1), (300, 20, 5, 2), (500, 37, 4, 2),
                                      (508, 64, 3, 4), (516, 16, 3, 1), (1000, 12, 3, 4), (1001, 1, 3, 2), (1024, 16, 3, 3)])
def test_sweep_with_weights_in_registers(ctx, H, mb, T, L):
    c = _case(H, mb, T, L)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 3)
    try:
        h, x, g, path, abandoned = _run(ctx, c)
        h2, x2, g2, _, _ = _run(ctx, c, times=3)  # flags of one launch must not reach the next
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 0)
    assert path == RESIDENT and not abandoned
    assert h.tobytes() == h2.tobytes() and x.tobytes() == x2.tobytes() and g.tobytes() == g2.tobytes()
    want_h, want_c = _want(c)
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")
    # the kept gates reproduce the states: c = clip(f c_prev + i c~), h = o tanh(c), 0 where masked
    m = (c["ids"] >= 0).astype(np.float32)[None, :, None, :]
    c_prev = np.concatenate([np.stack(c["c0"])[:, None], want_c[:, :-1]], axis=1)
    cell = np.clip(g[:, :, 1] * c_prev + g[:, :, 0] * g[:, :, 2], -0.9, 0.9)
    assert_close(m * cell, want_c, what="c from the gates")
    assert_close(m * g[:, :, 3] * np.tanh(cell), want_h, what="h from the gates")


@pytest.mark.parametrize("H,mb,T,L", [(100, 35, 6, 2), (100, 68, 5, 1), (300, 36, 6, 2), (500, 34, 5, 2), (500, 41, 5, 1),
                                      (500, 76, 4, 1)])
def test_back_to_back_with_different_inputs(ctx, H, mb, T, L):
    """Three and five column tiles of batches that are 1 to 4 columns beyond a multiple of eight, whose k-blocks in the
    hand-over copy would share cache lines were they padded to four columns: sweeps over different words and initial states
    queued one after another into the same scratch slots, so that a state left there by an earlier sweep is a wrong one."""
    cases = [_case(H, mb, T, L, seed=50 + i) for i in range(3)]
    for c in cases[1:]:
        c["layers"], c["embed"] = cases[0]["layers"], cases[0]["embed"]
    V, n = cases[0]["V"], H * mb
    layers, d_embed, runs = [Layer(ctx, ly) for ly in cases[0]["layers"]], ctx.array(cases[0]["embed"]), []
    for c in cases:
        d_nn, d_m = ctx.empty(c["ids"].size, np.int32), ctx.empty(c["ids"].size, np.int32)
        ctx.vocab_prep(ctx.array(c["ids"].reshape(-1)), c["ids"].size, V, d_nn, d_m)
        runs.append(dict(nn=d_nn, m=d_m, h0=[ctx.array(a) for a in c["h0"]], c0=[ctx.array(a) for a in c["c0"]],
                         h=[ctx.empty((n * T,)) for _ in range(L)], c=[ctx.empty((n * T,)) for _ in range(L)]))
    ctx.sync()
    try:
        for r in runs + runs[:2]:
            ctx.lstm_stack_forward([ly.w for ly in layers], d_embed, V, r["nn"], r["m"], T, mb, r["h0"], r["c0"], r["h"], r["c"])
            assert ctx.query(capi.ZR_QUERY_LSTM_SWEEP_KERNEL) == capi.ZR_LSTM_SWEEP_RESIDENT
        ctx.sync()
    finally:
        for ly in layers:
            ly.close()
    for i, (c, r) in enumerate(zip(cases, runs)):
        want_h, want_c = _want(c, clip=None)
        for got, want, what in ((r["h"], want_h, "h"), (r["c"], want_c, "c")):
            assert_close(np.stack([a.get().reshape(T, mb, H).swapaxes(1, 2) for a in got]), want, what="%s of sweep %d" % (what, i))


def test_library_picks_it_for_a_small_model(ctx):
    c = _case(100, 8, 5, 2)
    h, x, _, path, _ = _run(ctx, c)
    assert path == RESIDENT
    want_h, want_c = _want(c)
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")


def test_abandoned_wait_is_reported_and_leaves_nan(ctx):
    """With one poll per wait the upper layer gives up, every workgroup leaves, the outputs are NaN, and the next sweep
    with the default limit is complete again."""
    c = _case(100, 24, 6, 3)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 3)
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 1)
    try:
        h, x, g, path, abandoned = _run(ctx, c)
        assert path == RESIDENT and abandoned == 1
        assert np.all(np.isnan(h)) and np.all(np.isnan(x)) and np.all(np.isnan(g))
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
        h, x, g, path, abandoned = _run(ctx, c)
        assert path == RESIDENT and abandoned == 0
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 0)
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP_SPIN, 0)
    want_h, want_c = _want(c)
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")


# One node on tiles of 4 or 8 hidden rows (zr_lstm_rows.hip): row tails of every kind, columns around the edges of 16-, 32-
# and 64-column tiles, K tails of the last load (H % 4 and H % 8), with the embedding gather and with feed-input
@pytest.mark.parametrize("H,mb", [(8, 1), (9, 17), (11, 16), (100, 8), (127, 33), (130, 129), (257, 64), (500, 37), (510, 70),
                                  (513, 16), (1000, 12), (1000, 33), (1001, 130), (2000, 5)])
def test_node_on_narrow_row_tiles(ctx, H, mb):
    g = synth.rng(43, H + mb)
    V = 97
    ly = synth.lstm_layer(g, H, feed_input=True, forget_bias_one=True)
    embed = synth.uniform(g, (H, V), -0.5, 0.5)
    ids = g.integers(0, V, size=mb).astype(np.int32)
    hp, ht = np.tanh(synth.uniform(g, (H, mb), -1, 1)), np.tanh(synth.uniform(g, (H, mb), -1, 1))
    cp = synth.uniform(g, (H, mb), -0.5, 0.5)
    mask = (g.random(mb) < 0.8).astype(np.int32)
    layer = Layer(ctx, ly)
    d_h, d_c = ctx.empty((H, mb)), ctx.empty((H, mb))
    d_g = [ctx.empty((H, mb)) for _ in range(4)]
    x = np.asfortranarray(embed[:, ids])
    try:
        for feed in (False, True):
            want = o.lstm_step(ly["M"], ly["Wh"], ly["b"], x, hp, cp, mask, clip=0.9, **(dict(Q=ly["Q"], htild=ht) if feed else {}))
            for gather in (False, True):
                args = dict(clip=0.9, gates=d_g, d_htild=ctx.array(ht) if feed else None)
                if gather:
                    ctx.lstm_step_embed(layer.w, ctx.array(embed), V, ctx.array(ids), ctx.array(hp), ctx.array(cp),
                                        ctx.array(mask), mb, d_h, d_c, **args)
                else:
                    ctx.lstm_step(layer.w, ctx.array(x), ctx.array(hp), ctx.array(cp), ctx.array(mask), mb, d_h, d_c, **args)
                ctx.sync()
                what = "feed %d gather %d" % (feed, gather)
                assert_close(d_h.get(), want["h"], what="h " + what)
                assert_close(d_c.get(), want["c"], what="c " + what)
                for a, k in zip(d_g, ("i", "f", "c_tilde", "o")):
                    assert_close(a.get(), want[k], what=k + " " + what)
    finally:
        layer.close()


# ... and 4-row tiles beyond H = 512, two of which share the lines of the weights: odd numbers of them, the last size that has them
@pytest.mark.parametrize("H,mb", [(515, 1), (530, 16), (1021, 9), (1024, 16)])
def test_node_on_pairs_of_row_tiles(ctx, H, mb):
    test_node_on_narrow_row_tiles(ctx, H, mb)


# Infinite values where a k-group is only partly filled: beside an infinity nothing may be multiplied by a zero that stands
# for "not there".  H = 9, 100 and 101: the moved load of an embedding column's tail; 104: thirteen row tiles, whose last
# 16-column k-group is half empty; 300 at 40 columns: 32-column tiles.
@pytest.mark.parametrize("H,mb,L", [(9, 3, 1), (100, 8, 2), (101, 16, 1), (104, 8, 2), (300, 100, 1), (500, 12, 1), (1000, 12, 1)])
def test_sweep_with_infinite_inputs_saturates(ctx, H, mb, L):
    c = _case(H, mb, 4, L)
    words = np.unique(c["ids"][c["ids"] >= 0])
    for i, v in enumerate(words):  # at most one infinity a column: each gate's sum is then infinite and saturates
        if i % 3:
            c["embed"][H - 1 - (i % min(H, 6)), v] = np.inf if i % 2 else -np.inf
    c["h0"][0][H - 1, 0] = np.inf
    c["ids"][0, 0] = words[0]
    want_h, want_c = _want(c)
    assert np.isfinite(want_h).all() and np.isfinite(want_c).all()
    ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 3)
    try:
        h, x, _, path, _ = _run(ctx, c)
    finally:
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 0)
    assert path == RESIDENT
    assert_close(h, want_h, what="h")
    assert_close(x, want_c, what="c")


@pytest.mark.parametrize("H,mb", [(9, 3), (100, 8), (300, 20), (500, 12), (501, 37), (1000, 12), (1001, 70)])
def test_node_with_infinite_inputs_saturates(ctx, H, mb):
    g = synth.rng(47, H + mb)
    ly = synth.lstm_layer(g, H, forget_bias_one=True)
    x, hp = synth.uniform(g, (H, mb), -0.5, 0.5), np.tanh(synth.uniform(g, (H, mb), -1, 1))
    cp, mask = synth.uniform(g, (H, mb), -0.5, 0.5), np.ones(mb, np.int32)
    x[H - 1, 0], hp[H - 2, 1] = np.inf, -np.inf
    for gate in range(4):
        ly["M"][gate][H // 2, H - 1] = np.inf   # infinite weights meet column 0's infinity with one sign only
        ly["Wh"][gate][H // 2 - 1, H - 3] = -np.inf
    x[H - 1, 2:] = 0.25
    want = o.lstm_step(ly["M"], ly["Wh"], ly["b"], x, hp, cp, mask)
    fine = np.isfinite(want["h"])
    assert fine.mean() > 0.85
    layer = Layer(ctx, ly)
    d_h, d_c = ctx.empty((H, mb)), ctx.empty((H, mb))
    try:
        ctx.lstm_step(layer.w, ctx.array(x), ctx.array(hp), ctx.array(cp), ctx.array(mask), mb, d_h, d_c)
        ctx.sync()
    finally:
        layer.close()
    assert np.array_equal(np.isfinite(d_h.get()), fine)
    assert_close(np.where(fine, d_h.get(), 0), np.where(fine, want["h"], 0), what="h")
    assert_close(np.where(fine, d_c.get(), 0), np.where(fine, want["c"], 0), what="c")


def _sigmoid(v):
    return 1.0 / (1.0 + np.exp(-v))


def _cell_in_64_bits(z, c):
    zi, zf, zc, zo = np.split(z, 4)
    c = _sigmoid(zf) * c + _sigmoid(zi) * np.tanh(zc)
    return _sigmoid(zo) * np.tanh(c), c


def _wide(layer, key):
    return np.concatenate([np.asarray(a, np.float64).reshape(layer["b"][0].size, -1) for a in layer[key]])


def _rough_layer(g, H, **kw):
    """Weights large enough that the products' rounding is most of the error of h."""
    layer = synth.lstm_layer(g, H, **kw)
    return {k: [synth.uniform(g, a.shape, -1.5 / H ** 0.5, 1.5 / H ** 0.5) for a in v] for k, v in layer.items()}


# one size of every form whose sums go through LDS in pieces or have two accumulators, where the launches per diagonal divide K
@pytest.mark.parametrize("H,mb", [(200, 16), (400, 8), (512, 16), (768, 1), (768, 40), (1000, 16), (1024, 8), (1024, 40)])
def test_sweep_rounds_no_more_than_one_launch_per_diagonal(ctx, H, mb):
    """The two schedules' errors against 64 bits, each an average over T * H * mb values.  How they vary between draws of that
    size is a few per cent; one chain of additions a wave was 1.25 (H = 512) to 1.6 times (1024) the other schedule's error."""
    g, T, V = synth.rng(47, H + mb), 12, 300
    c = dict(H=H, mb=mb, T=T, L=1, V=V, ids=g.integers(0, V, size=(T, mb)).astype(np.int32),
             embed=synth.uniform(g, (H, V), -1, 1), layers=[_rough_layer(g, H)], h0=[np.zeros((H, mb), np.float32)],
             c0=[np.zeros((H, mb), np.float32)])
    M, W, b = [_wide(c["layers"][0], k) for k in ("M", "Wh", "b")]
    want, hp, cp = [], np.zeros((H, mb)), np.zeros((H, mb))
    for t in range(T):
        hp, cp = _cell_in_64_bits(M @ c["embed"][:, c["ids"][t]].astype(np.float64) + W @ hp + b, cp)
        want.append(hp)
    error = {}
    for option in (1, 3):
        ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, option)
        try:
            h, _, _, path, _ = _run(ctx, c, clip=0.0)
        finally:
            ctx.set_option(capi.ZR_OPT_LSTM_SWEEP, 0)
        assert (path == RESIDENT) == (option == 3)
        error[option] = np.linalg.norm(h[0] - np.stack(want)) / np.linalg.norm(want)
    assert error[3] < 1.1 * error[1]


# 4 x 16, 8 x 16, 8 x 32 and 8 x 64 tiles with and without feed-input
@pytest.mark.parametrize("H,mb", [(500, 37), (512, 8), (1000, 16), (1024, 1), (1024, 40), (1200, 8), (500, 128)])
@pytest.mark.parametrize("feed", [False, True])
def test_node_is_rounded_in_short_chains(ctx, H, mb, feed):
    """Error of the pre-activations against 64 bits, from c' = f c + i u with c = 0 and i near 1 (a bias of 20): u = tanh(z_c), z_c
    small, carries z_c's.  An addition rounds its result by a relative 2.5e-8 in the 2-norm, a chain of n by sqrt(n / 2) of
    that; each wave's K / 8 products are four chains in 8 x 16 tiles, else two; then the chains and the
    waves' sums are added pairwise (five additions of at most the final size).  A third above that passes: i, u and c' round too."""
    g = synth.rng(48, H + mb)
    layer = _rough_layer(g, H, feed_input=feed)
    layer["M"][2], layer["Wh"][2] = layer["M"][2] * 0.02, layer["Wh"][2] * 0.02
    if feed:
        layer["Q"][2] = layer["Q"][2] * 0.02
    layer["b"][0][:], layer["b"][2][:] = 20.0, 0.0
    ly = Layer(ctx, layer)
    x, hp, ht = [synth.uniform(g, (H, mb), -1, 1) for _ in range(3)]
    d_h, d_c, ones = ctx.empty((H, mb)), ctx.empty((H, mb)), ctx.array(np.ones(mb, np.int32))
    try:
        if feed:
            ids = ctx.array(np.arange(mb, dtype=np.int32))
            ctx.lstm_step_embed(ly.w, ctx.array(x), mb, ids, ctx.array(hp), ctx.zeros((H, mb)), ones, mb, d_h, d_c, d_htild=ctx.array(ht))
        else:
            ctx.lstm_step(ly.w, ctx.array(x), ctx.array(hp), ctx.zeros((H, mb)), ones, mb, d_h, d_c)
        ctx.sync()
    finally:
        ly.close()
    z = np.asarray(layer["M"][2], np.float64) @ x + np.asarray(layer["Wh"][2], np.float64) @ hp
    if feed:
        z += np.asarray(layer["Q"][2], np.float64) @ ht
    want = np.tanh(z)
    K = (3 if feed else 2) * H
    n = K / 8 / (4 if H > 512 and (mb <= 16 or (H + 7) // 8 * ((mb + 15) // 16) <= 256) else 2)
    error = np.linalg.norm(d_c.get() - want) / np.linalg.norm(want)
    assert error < 1.33 * 2.5e-8 * np.sqrt(n / 2 + 5)
