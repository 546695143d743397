"""The attention node's backward pass over batches whose sums over the columns are made in parts (zr_attn_sum_parts), at its line and with
a last part of one column, hidden sizes off the 32-row blocks."""
import pytest

from test_gpu_backward import ctx  # noqa: F401
from test_gpu_backward import test_attention_backward_against_oracle as against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,mb,S,D", [(33, 512, 4, 2), (48, 513, 5, 2), (70, 769, 3, 1), (31, 1030, 4, 3)])
def test_wide_batches(ctx, H, mb, S, D):  # noqa: F811
    against_oracle(ctx, H, mb, S, D)
