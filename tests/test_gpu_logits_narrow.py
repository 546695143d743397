"""The output layer's product on a prepared fp32 matrix for up to 16 columns (csrc/zr_logits_narrow.hip): edges of its 16-row tiles and 32-row blocks, of its
groups of 16 k and their ring, both forms, and activations that are infinite; and the split product's one 32-column block at 17 to 32 columns.  Tolerance: H products and their sums, each rounded
once (test_gpu_logits_split.py's bound; the eight chains round less)."""
import numpy as np
import pytest

from test_gpu_logits_split import bound, logits_and_blocks, operands
from zoph_rnn_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def check(D, b, h, x, pairs):
    V, n = x.shape
    assert np.all(np.abs(x - (D.astype(np.float64) @ h + b[:, None])) <= bound(D, b, h))
    pad = np.full(((V + 31) // 32 * 32, n), -np.inf)
    pad[:V] = x
    pad = pad.reshape((-1, 32, n))
    assert np.array_equal(pairs[:, :, 0], pad.max(axis=1).T.astype(np.float32))
    want = np.exp(pad - pad.max(axis=1, keepdims=True)).sum(axis=1).T
    assert np.all(np.abs(pairs[:, :, 1] - want) <= 64 * 2.0 ** -24 * want)


@pytest.mark.parametrize("V,H,n", [(1, 4, 1), (15, 5, 3), (16, 7, 16), (31, 8, 2), (33, 15, 15), (63, 16, 4), (64, 17, 16), (65, 31, 1), (100, 64, 9), (129, 65, 16), (1000, 80, 13),
                                   (4097, 333, 12), (8191, 640, 5), (9000, 1000, 16), (10001, 81, 7), (30011, 500, 12), (49152, 12, 16), (50001, 20, 3), (50000, 96, 12),
                                   (65536, 33, 2), (65537, 8, 1), (50001, 400, 11), (20011, 1003, 10)])
def test_logits_and_block_pairs(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    check(D, b, h, *logits_and_blocks(ctx, D, b, h))


@pytest.mark.parametrize("V,H,n", [(45568, 401, 2), (45569, 400, 12), (50001, 417, 3), (48900, 1003, 16), (65505, 402, 1), (65536, 399, 5), (65536, 401, 16), (65537, 404, 7)])
def test_four_waves_of_64_rows_around_their_line(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    check(D, b, h, *logits_and_blocks(ctx, D, b, h))


@pytest.mark.parametrize("V,H,n", [(125, 536, 9), (2047, 512, 3), (2048, 512, 5), (2048, 513, 16), (4001, 600, 2), (4001, 608, 12), (8191, 555, 7), (8192, 601, 12), (8193, 601, 2)])
def test_few_rows_of_a_long_k(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    check(D, b, h, *logits_and_blocks(ctx, D, b, h))


@pytest.mark.parametrize("V,H,n", [(1, 1, 17), (33, 31, 31), (257, 128, 32), (8192, 200, 18), (8449, 264, 32), (10001, 63, 25), (20480, 1000, 17), (30011, 500, 32), (33333, 333, 29),
                                   (50001, 96, 24)])
def test_one_block_of_columns(ctx, V, H, n):
    D, b, h = operands(V, H, n)
    check(D, b, h, *logits_and_blocks(ctx, D, b, h))


@pytest.mark.parametrize("V,H", [(50001, 20), (9001, 37)])
def test_infinite_activations_stay_in_their_columns(ctx, V, H):
    D, b, h = operands(V, H, 5)
    h[H - 1, 2] = np.inf
    x, pairs = logits_and_blocks(ctx, D, b, h)
    assert np.array_equal(x[:, 2], np.where(D[:, H - 1] > 0, np.inf, -np.inf).astype(np.float32))
    keep = [0, 1, 3, 4]
    check(D, b, np.asfortranarray(h[:, keep]), x[:, keep], pairs[keep])


def test_an_infinite_weight_stays_in_its_row(ctx):
    D, b, h = operands(9000, 37, 6)
    D[4321, 36] = np.inf
    x, _ = logits_and_blocks(ctx, D, b, h)
    assert np.array_equal(x[4321], np.where(h[36] > 0, np.inf, -np.inf).astype(np.float32))
    assert np.all(np.isfinite(np.delete(x, 4321, axis=0)))
