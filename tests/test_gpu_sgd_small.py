"""The clipped update of a matrix in one launch (sgd_small_kernel) around its block sizes, its limit and off 16-byte alignment.
Tolerance: the factor's product, square root, quotient and two multiplications, 2^-24 each, times the step; one rounding of the step and one
of the sum."""
import ctypes

import numpy as np
import pytest
import torch

from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1025, 4096, 4099, 16385, 27999, 28001, 65537, 111999, 112000, 112001])
@pytest.mark.parametrize("off_w,off_g", [(0, 0), (1, 0), (4, 2)])
@pytest.mark.parametrize("clip", [0.5, 1e6])
def test_update(ctx, n, off_w, off_g, clip):
    r = np.random.default_rng(n + off_w + 8 * off_g)
    w, g = r.uniform(-1, 1, n + 8).astype(np.float32), r.normal(0, 3, n + 8).astype(np.float32)
    dw, dg = ctx.array(w), ctx.array(g)
    scale, lr = 0.05, 0.7
    ctx.sgd_update(dw.at(off_w), dg.at(off_g), n, scale, clip, lr)
    ctx.sync()
    x = g[off_g:off_g + n].astype(np.float64) * np.float32(scale)
    norm = np.linalg.norm(x)
    step = np.float32(lr) * x * (min(1.0, np.float32(clip) / norm) if norm else 1.0)
    want = w.astype(np.float64)
    want[off_w:off_w + n] += step
    got = dw.get()
    assert np.array_equal(np.delete(got, np.s_[off_w:off_w + n]), np.delete(w, np.s_[off_w:off_w + n]))
    assert np.all(np.abs(got - want)[off_w:off_w + n] <= 2.0 ** -24 * (7 * np.abs(step) + np.abs(want[off_w:off_w + n])))


def test_non_finite_gradient_reaches_every_value(ctx):
    g = np.ones(5000, np.float32)
    g[4321] = np.nan
    dw = ctx.array(np.ones(5000, np.float32))
    ctx.sgd_update(dw, ctx.array(g), 5000, 1.0, 5.0, 0.1)
    ctx.sync()
    # a norm that is no number is not above the threshold: the other values take the plain step
    want = np.where(np.isnan(g), np.nan, np.float32(1) + np.float32(0.1))
    assert np.array_equal(dw.get(), want.astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("n", [27999, 28001, 65537, 112000, 112001, 250001])
@pytest.mark.parametrize("off_w,off_g", [(0, 0), (1, 0)])
def test_update_on_a_callers_stream(n, off_w, off_g):
    """Where the workgroups' sums cannot be exchanged: this kernel to its limit, then two launches."""
    c = capi.Context(0)
    s = torch.cuda.Stream()
    capi._chk(capi.load().zr_ctx_set_stream(c.h, ctypes.c_void_p(s.cuda_stream)))
    test_update(c, n, off_w, off_g, 0.5)
    capi._chk(capi.load().zr_ctx_set_stream(c.h, None))
    c.close()
