"""The output layer's product on a prepared bf16 matrix for up to 64 columns (csrc/zr_logits_bf16.hip): edges of its 32-row blocks and 128-row workgroups, of
its chunks of 64 k and their ring, one and two 32-column blocks, one and two activation terms.  The matrix is exact in bf16, with one term the activations too.
Tolerance: at most 2 H products and their sums, each rounded once (test_gpu_logits_split.py's bound, twice with two terms), and with two terms
2^-18 of every product for the activations' own rounding."""
import numpy as np
import pytest

from test_gpu_logits_split import bound, operands
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 2])
def ctx(request):
    c = capi.Context(0)
    c.set_option(capi.ZR_OPT_BF16_ACTIVATION_TERMS, request.param)
    c.terms = request.param
    yield c
    c.close()


def bf16(x):
    u = x.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("V,H,n", [(10000, 16, 1), (10001, 48, 2), (10015, 64, 33), (10016, 80, 63), (10017, 128, 64), (10111, 144, 16), (10112, 192, 17), (10113, 208, 31),
                                   (10143, 336, 37), (10144, 528, 64), (20000, 1024, 48), (30011, 400, 12), (33333, 1040, 64), (70001, 480, 1), (65537, 528, 32),
                                   (50000, 1008, 33), (12345, 256, 64)])
def test_logits_and_block_pairs(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    D = bf16(D)
    if ctx.terms == 1:
        h = bf16(h)
    blocks, off = (V + 31) // 32, (V * n + 3) // 4 * 4
    dD = ctx.array(D)
    ctx.softmax_prepare(dD, V, H, bf16=True)
    out = ctx.array(np.full(off + 2 * blocks * n + 1, 7.0, np.float32))
    ctx.softmax_forward(dD, ctx.array(b), V, H, ctx.array(h), n, capi.ZR_SOFTMAX_LOGITS_BLOCKS, out)
    ctx.sync()
    ctx.softmax_release(dD)
    o = out.get()
    assert o[-1] == 7.0
    x, pairs = o[:V * n].reshape((V, n), order="F"), o[off:-1].reshape((n, blocks, 2))
    rounding = 0.0 if ctx.terms == 1 else 2.0 ** -18 * (np.abs(D).astype(np.float64) @ np.abs(h))
    assert np.all(np.abs(x - (D.astype(np.float64) @ h + b[:, None])) <= ctx.terms * bound(D, b, h) + rounding)
    pad = np.full((blocks * 32, n), -np.inf)
    pad[:V] = x
    pad = pad.reshape((-1, 32, n))
    assert np.array_equal(pairs[:, :, 0], pad.max(axis=1).T.astype(np.float32))
    want = np.exp(pad - pad.max(axis=1, keepdims=True)).sum(axis=1).T
    assert np.all(np.abs(pairs[:, :, 1] - want) <= 64 * 2.0 ** -24 * want)
