"""The output projection that holds its weights in registers (gemm_resident_kernel.h), which the attention layer takes up to 112 rows:
a row, one short of sixteen rows, sixteen, one more, two, four and seven groups of rows; K that leaves wavefronts without a share, with a
ragged last one and with all of it; columns that end inside a workgroup's.  Every mode against the oracle on the GPU's own
intermediates and against stream order bit for bit."""
import pytest

import test_gpu_attention as attention
from cusync_amd import api

pytestmark = pytest.mark.gpu


def grid3(S, hidden, heads, **kw):
    """The third stage's grid of a layer that is made and not run."""
    _, _, dwqkv, dwo = attention.layer_weights(hidden, heads)
    layer = api.AttnLayer(S, hidden, heads, api.SYNC.ROW, dwqkv.data_ptr(), dwo.data_ptr(), **kw)
    grid = layer.stage_state(2).grid
    layer.destroy()
    return tuple(grid)


def grids(hidden):
    return [((hidden + n - 1) // n, 1, 1) for n in (64, 128)]


@pytest.mark.parametrize("S,hidden,heads", [(1, 8192, 12), (15, 8192, 1), (16, 8152, 3), (17, 8200, 5), (32, 8192, 11), (33, 8192, 12), (64, 8152, 12),
                                            (48, 16384, 3), (64, 12288, 12), (65, 8192, 12), (112, 8152, 12)])
def test_layer_matches_oracle(S, hidden, heads):
    print("resident", S, hidden, heads, flush=True)
    assert grid3(S, hidden, heads) in grids(hidden)
    attention.check_layer(S, hidden, heads, sampled=False)


# 64 columns to a workgroup where each has a CU beside the attention's, 128 where the cache brings that more workgroups, and in
# stream order always 64; the few-row attention's tiles and the 128-row tiles of the general one in front of it
def test_columns_of_a_workgroup():
    assert grid3(16, 12288, 12) == grids(12288)[0] and grid3(16, 12288, 12, cached_rows=2048) == grids(12288)[1]


@pytest.mark.parametrize("S,cached", [(1, 130), (16, 2048), (32, 300), (33, 700), (64, 64), (100, 1000), (112, 2000)])
def test_layer_with_cache(S, cached):
    print("resident behind", S, cached, flush=True)
    attention.test_attention_layer_with_cache(S, cached)


@pytest.mark.parametrize("S,hidden,heads,kw", [(113, 8192, 12, {}), (16, 8064, 12, {}), (16, 8192, 13, {}),
                                               (16, 8192, 12, {"tile3": api.TILE.D32x128x64}), (16, 8192, 12, {"opts": api.OPT.AVOID_WAIT_KERNEL})])
def test_tiles_outside_its_range(S, hidden, heads, kw):
    print("not resident", S, hidden, heads, kw, flush=True)
    assert grid3(S, hidden, heads, **kw) not in grids(hidden)
