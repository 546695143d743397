"""Products large enough for the bf16 matrix cores with every fp32 operand as three bf16 terms, and what feeds them.  (The forward product of a prepared
output layer here is zr_logits.hip's; the split product takes one from 4 GiB on, tests/test_gpu_logits_split.py.)"""
import numpy as np
import pytest

from zoph_rnn_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def rel(got, want):
    return np.linalg.norm(np.asarray(got, np.float64) - want) / np.linalg.norm(want)


def bound(K):
    # An element is a chain of 6 fp32 additions per 16 k, each rounding a partial sum of at most the final size (in the
    # 2-norm over random operands) by 2^-24; independent roundings add in squares.  One missing term of an operand would
    # be 2^-17 and more.
    return 2.0 ** -24 * np.sqrt(6 * K / 16)


# edges of the 128 x 128 and 128 x 256 tiles and of the 32-k steps, K in parts, operands at odd leading dimensions
@pytest.mark.parametrize("M,N,K,pad", [(1024, 1024, 1024, 0), (1025, 1001, 1003, 1), (257, 256, 16000, 0), (259, 513, 8191, 3),
                                       (16001, 257, 256, 2), (8192, 300, 509, 0)])
@pytest.mark.parametrize("trans", [0, 1])
def test_gemm(ctx, M, N, K, pad, trans):
    g = synth.rng(41, M + N)
    A = np.zeros(((K if trans else M) + pad, M if trans else K), np.float32, order="F")
    A[:K if trans else M] = g.standard_normal((K, M) if trans else (M, K)).astype(np.float32)
    B = np.full((K + pad, N), np.nan, np.float32, order="F")
    B[:K] = g.standard_normal((K, N)).astype(np.float32)
    A[K if trans else M:] = np.nan
    dC = ctx.array(np.full((M + pad, N), 7.0, np.float32, order="F"))
    ctx.gemm(trans, M, N, K, ctx.array(A), A.shape[0], ctx.array(B), K + pad, dC, M + pad)
    ctx.sync()
    a = (A[:K].T if trans else A[:M]).astype(np.float64)
    C = dC.get()
    assert rel(C[:M], a @ B[:K].astype(np.float64)) < bound(K)
    assert np.all(C[M:] == 7.0)


def test_gemm_keeps_all_24_bits_and_small_values(ctx):
    """One term per sum: the product of two 24-bit values.  Sizes down to 2^-35 per operand (times a normal variate, seldom
    below 2^-10): the smallest of the six products, 2^-16 of the result, stays a normal number (above 2^-126)."""
    g = synth.rng(42, 1)
    n = 1024
    A = np.zeros((n, n), np.float32, order="F")
    np.fill_diagonal(A, (g.standard_normal(n) * 2.0 ** g.integers(-35, 30, n)).astype(np.float32))
    B = np.asfortranarray((g.standard_normal((n, n)) * 2.0 ** g.integers(-35, 30, (n, n))).astype(np.float32))
    dC = ctx.empty((n, n))
    ctx.gemm(0, n, n, n, ctx.array(A), n, ctx.array(B), n, dC, n)
    ctx.sync()
    want = np.diag(A).astype(np.float64)[:, None] * B.astype(np.float64)
    # the six products are added one by one: three half units in the last place and what the three left out hold
    assert np.max(np.abs(dC.get() / want - 1.0)) < 4 * 2.0 ** -24


def test_gemm_infinities_and_nan(ctx):
    g = synth.rng(43, 1)
    n = 1024
    A = np.asfortranarray(g.standard_normal((n, n)).astype(np.float32))
    B = np.asfortranarray(g.standard_normal((n, n)).astype(np.float32))
    A[5, 17], A[700, 900], A[701, 3], A[130, 44] = np.inf, -np.inf, np.nan, 3.4e38  # the last rounds to infinity in bf16
    B[44] *= 1e-3
    B[17, 9], B[900, 30], B[64, 1000] = 0.0, np.inf, 1.0
    dC = ctx.empty((n, n))
    ctx.gemm(0, n, n, n, ctx.array(A), n, ctx.array(B), n, dC, n)
    ctx.sync()
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    got = dC.get()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    fine = np.isfinite(want)
    rows = np.arange(n) != 130
    assert np.all(np.isfinite(got[fine]))
    assert rel(got[rows][fine[rows]], want[rows][fine[rows]]) < bound(n)
    assert rel(got[130][fine[130]], want[130][fine[130]]) < bound(n)


@pytest.mark.parametrize("V,H,n,prepared", [(9001, 260, 520, True), (9001, 260, 520, False), (4133, 500, 1100, True),
                                            (12000, 333, 257, True),
                                            # the error pass with 2 columns a workgroup (a last chunk of one) and with 16
                                            (1000, 64, 33, False), (1003, 30, 2, False), (1000, 100, 1000, True),
                                            (4097, 52, 1001, False)])
def test_output_layer(ctx, V, H, n, prepared):
    g = synth.rng(44, V + n)
    D = synth.uniform(g, (V, H), -0.2, 0.2)
    bd, h = synth.uniform(g, (V,), -1, 1), synth.uniform(g, (H, n), -1, 1)
    target, mask = g.integers(0, V, size=n).astype(np.int32), (g.random(n) > 0.2).astype(np.int32)
    x = D.astype(np.float64) @ h.astype(np.float64) + bd.astype(np.float64)[:, None]
    x -= np.log(np.exp(x).sum(0))
    dD, db, dh, dt, dm = ctx.array(D), ctx.array(bd), ctx.array(h), ctx.array(target), ctx.array(mask)
    if prepared:
        ctx.softmax_prepare(dD, V, H)
    scr, eh, gD, gb = ctx.empty((V, n)), ctx.empty((H, n)), ctx.empty((V, H)), ctx.empty((V,))
    ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_LOGPROB, scr)
    ctx.sync()
    assert np.max(np.abs(scr.get() - x)) < 2e-5  # logits of size 10 in fp32: 2^-21 each and the sum's part
    want = float((x[target, np.arange(n)] * mask).sum())
    assert ctx.softmax_loss(dD, db, V, H, dh, n, dt, dm, scr) == pytest.approx(want, rel=1e-6)
    for accumulate in (False, True):
        loss = None
        if accumulate:
            ctx.softmax_backward(dD, db, V, H, dh, n, dt, dm, scr, eh, gD, gb, accumulate=True)
            ctx.sync()
        else:
            loss = ctx.softmax_backward_loss(dD, db, V, H, dh, n, dt, dm, scr, eh, gD, gb)
            assert loss == pytest.approx(want, rel=1e-6)
        e = -np.exp(x)
        e[target, np.arange(n)] += 1.0
        e *= mask
        times = 2.0 if accumulate else 1.0
        # every e carries the rounding of its logit, 10 * 2^-24 relative, beside the sums' own
        assert rel(scr.get(), e) < 2e-6
        assert rel(eh.get(), D.T.astype(np.float64) @ e) < 2e-6 + bound(V)
        assert rel(gD.get(), times * (e @ h.T.astype(np.float64))) < 2e-6 + bound(n)
        assert rel(gb.get(), times * e.sum(1)) < 4e-6
        assert np.all(eh.get()[:, mask == 0] == 0)
    if prepared:
        ctx.softmax_release(dD)


@pytest.mark.parametrize("H,T,mb", [(300, 30, 100), (513, 1, 1200), (260, 61, 67)])
def test_lstm_weight_gradients(ctx, H, T, mb):
    g = synth.rng(45, H)
    K = T * mb
    dg, x, h = (g.standard_normal(s).astype(np.float32, order="F") for s in ((4 * H, K), (H, K), (H, K)))
    h0 = g.standard_normal((H, mb)).astype(np.float32, order="F")
    dM, dWh, db = ctx.empty((4 * H, H)), ctx.empty((4 * H, H)), ctx.empty((4 * H,))
    ctx.lstm_weight_gradients(H, T, mb, ctx.array(dg), ctx.array(x), ctx.array(h0), ctx.array(h), dM, dWh, db)
    ctx.sync()
    prev = np.concatenate([h0, h[:, :K - mb]], 1).astype(np.float64)
    d = dg.astype(np.float64)
    assert rel(dM.get(), d @ x.T.astype(np.float64)) < bound(K)
    assert rel(dWh.get(), d @ prev.T) < bound(K)
    assert rel(db.get(), d.sum(1)) < bound(K)


@pytest.mark.parametrize("V,H,n", [(20000, 500, 257), (20001, 503, 512), (10001, 1000, 400), (12000, 1000, 1024)])
def test_prepared_output_layer_is_rounded_in_short_chains(ctx, V, H, n):
    """With sums of 32 k (zr_logits.hip; a bound for 16).  A probability is off by its logit's error, in proportion.  The logit of a large one is a sum that grows steadily, so the
    partial sums have a third of the final square on average: K / 16 additions, each a relative 2.5e-8 in the 2-norm (mantissas
    spread evenly in their logarithm), and the bias.  The exponential, its argument, the sum and the division add a part in
    10^7.  (Measured: two thirds of that.  With the six products of 16 k added one by one twice to three times as much.)"""
    g = synth.rng(46, V + n)
    D = g.standard_normal((V, H)).astype(np.float32) / np.float32(H ** 0.5 / 3)
    b = g.standard_normal(V).astype(np.float32)
    h = g.standard_normal((H, n)).astype(np.float32)
    dD, db, dh, out = ctx.array(np.asfortranarray(D)), ctx.array(b), ctx.array(np.asfortranarray(h)), ctx.empty((V, n))
    ctx.softmax_prepare(dD, V, H)
    try:
        ctx.softmax_forward(dD, db, V, H, dh, n, capi.ZR_SOFTMAX_PROB, out)
        ctx.sync()
    finally:
        ctx.softmax_release(dD)
    z = D.astype(np.float64) @ h + b[:, None]
    p = np.exp(z - z.max(0))
    p /= p.sum(0)
    size = np.sqrt((p * p * z * z).sum() / (p * p).sum())  # of the logits that count
    error = np.linalg.norm(out.get() - p) / np.linalg.norm(p)
    assert error < size * 2.5e-8 * np.sqrt(H / 16 / 3) + 1e-7
