"""The attention kernel of up to 32 query rows with a split key range, at the edges of its range."""
import numpy as np
import pytest

import oracle as orc
from test_gpu_attention import run_attention_split
from util import assert_close, normal_f16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
# one key more than a piece, a piece of new rows only, splits that leave wavefronts without keys, more than eight
# splits (read back in two groups), the largest row count of the kernel and the first of the other one
@pytest.mark.parametrize("S,cached,heads,blocks", [(1, 64, 1, 1), (1, 96, 2, 1), (32, 33, 1, 1), (31, 130, 3, 2), (32, 1000, 1, 1),
                                                   (5, 1100, 2, 2), (16, 2048, 12, 6), (33, 300, 1, 2)])
def test_few_rows_split_key_range(S, cached, heads, blocks, causal):
    print("attention few", S, cached, heads, blocks, causal, flush=True)
    qkv = normal_f16((cached + S, 3 * heads * 128), 31, std=1.0)
    got, grid = run_attention_split(qkv, cached, heads, causal, blocks)
    assert grid == (heads, 1, -(-(-(-(cached + S) // 64)) // blocks))
    assert_close(got, orc.attention_kv(qkv, cached, heads, 128, causal), "O")
    one, _ = run_attention_split(qkv, cached, heads, causal, blocks, launches=1, max_workgroups=1)
    assert np.array_equal(got.view(np.uint16), one.view(np.uint16))       # the result does not depend on arrival order
