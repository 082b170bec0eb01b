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


def reference(qkv, cached, heads, scale):
    """Causal attention in float64, the result rounded to halfs."""
    q, k, v = (qkv[:, i * heads * 128:(i + 1) * heads * 128].reshape(-1, heads, 128).transpose(1, 0, 2).astype(np.float64) for i in range(3))
    s = (q[:, cached:] @ k.transpose(0, 2, 1)) * (scale or 128 ** -0.5)
    s[:, ~np.tri(s.shape[1], s.shape[2], cached, dtype=bool)] = -np.inf
    p = np.exp(s - s.max(axis=2, keepdims=True))
    return ((p / p.sum(axis=2, keepdims=True)) @ v).transpose(1, 0, 2).reshape(-1, heads * 128).astype(np.float16)


# Keys a query does not see, where they are all that a wavefront's first piece (up to 32 rows) or a split's first block
# (more rows: the splits begin inside the new rows) holds for it: nothing may come of them at any scale.
@pytest.mark.parametrize("scale", [0.0, 0.125, 0.0625, 0.05, 1.0, 4.0])
@pytest.mark.parametrize("S,cached,heads,blocks", [(32, 2000, 1, 1), (32, 33, 1, 1), (32, 84, 2, 1), (17, 300, 3, 2),
                                                   (128, 20, 1, 1), (130, 0, 2, 1), (300, 70, 1, 2)])
def test_masked_keys_weigh_nothing(S, cached, heads, blocks, scale):
    print("attention masked", S, cached, heads, blocks, scale, flush=True)
    qkv = normal_f16((cached + S, 3 * heads * 128), 33, std=1.0)
    got, grid = run_attention_split(qkv, cached, heads, True, blocks, scale=scale)
    assert grid[2] > 1
    assert_close(got, reference(qkv, cached, heads, scale), "O")
