"""The attention kernel of up to 32 query rows with a split key range, at the edges of its range."""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
import test_gpu_attention as attention
from cusync_amd import _lib, api
from test_gpu_attention import run_attention_split
from util import assert_close, empty_dev, normal_f16, to_dev, to_host, uniform_f16

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


def test_few_rows_of_a_stage_that_may_start_last():
    """Under AvoidWaitKernel a stage that is no larger than its caller counted on: bit for bit the kernel of more rows, whose
    last 17 of 33 these are."""
    import torch
    print("attention few AvoidWaitKernel", flush=True)
    heads, total, blocks = 3, 317, 1
    qkv = normal_f16((total, 3 * heads * 128), 35, std=1.0)
    dq, outs = to_dev(qkv), {}
    # a stage that posts (to nobody), so that it is not alone on its stream
    post = api.tile_sync(api.ORDER.TRANSPOSE_XY, 128, 128)
    for S, opts in ((17, api.OPT.AVOID_WAIT_KERNEL), (33, 0), (17, 0)):
        cached = total - S
        o = empty_dev((S, heads * 128), fill=float("nan"))
        ws = torch.zeros(api.attention_workspace_size(S, heads, cached, blocks), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        st = api.Stage(api.attention_grid(S, heads, cached, blocks), (1, 1, 1), api.no_sync(), post, opts=opts)
        assert api.attention(st, S, heads, dq.data_ptr(), 3 * heads * 128, o.data_ptr(), heads * 128, cached_rows=cached,
                             kv_split_blocks=blocks, workspace=ws.data_ptr()) == api.ERR.SUCCESS, api.last_error()
        torch.cuda.synchronize()
        st.destroy()
        outs[S, opts] = to_host(o)
        assert_close(outs[S, opts], orc.attention_kv(qkv, cached, heads, 128, True), "O")
    assert np.array_equal(outs[17, api.OPT.AVOID_WAIT_KERNEL].view(np.uint16), outs[33, 0][16:].view(np.uint16))


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


# as the second stage of the chain under every policy, with a piece that holds cached and new rows
@pytest.mark.parametrize("S,cached", [(7, 130), (17, 300), (32, 2031)])
def test_few_rows_in_the_layer(S, cached):
    attention.test_attention_layer_with_cache(S, cached)


@pytest.mark.parametrize("sync", ["row", "tile", "consecutive"])
@pytest.mark.parametrize("S,cached,blocks,more", [(17, 300, 1, 0), (17, 300, 1, 8), (32, 2031, 6, 8), (1, 130, 1, 8)])
def test_few_rows_behind_a_projection(S, cached, blocks, more, sync):
    """A consumer that reads the cached rows before it waits.  With a row pitch or a base that is not whole 128-byte lines
    (`more` halfs) the last cached row shares a line with the first new one, which the wait then has to invalidate."""
    import torch
    print("attention few consumer", S, cached, blocks, more, sync, flush=True)
    L = _lib.load()
    hidden, heads, tile = 4096, 3, api.TILE.D32x128x64
    E, ld = heads * 128, 3 * heads * 128 + more
    w = normal_f16((hidden, 3 * E), 41)
    xs = [uniform_f16((S, hidden), 42 + r) for r in range(3)]
    cache = normal_f16((cached, 3 * E), 40, std=1.0)
    flat = torch.full((more + (cached + S) * ld,), float("nan"), dtype=torch.float16, device="cuda")
    qkv = flat[more:].view(cached + S, ld)
    qkv[:cached, :3 * E] = to_dev(cache)
    o, dw, dxs = empty_dev((S, E)), to_dev(w), [to_dev(x) for x in xs]
    tm, tn, _ = api.tile_shape(tile)
    grid = api.gemm_grid(tile, S, 3 * E)
    pol = {"row": api.row_sync(tm, grid[0]), "tile": api.tile_sync(api.ORDER.TRANSPOSE_XY, tm, tn),
           "consecutive": api.consecutive_sync(api.ORDER.TRANSPOSE_XY, 8 * E, tm, tn)}[sync]
    prod = api.Stage(grid, (1, 1, 1), api.no_sync(), pol)
    cons = api.Stage(api.attention_grid(S, heads, cached, blocks), (1, 1, 1), pol, api.no_sync())
    assert cons.grid()[2] > 1 and api.set_producer_consumer_pair(prod, cons) == api.ERR.SUCCESS
    ws = torch.zeros(api.attention_workspace_size(S, heads, cached, blocks), dtype=torch.uint8, device="cuda")
    s0, s1 = torch.cuda.Stream(), torch.cuda.Stream()
    for x, dx in zip(xs, dxs):
        qkv[cached:] = float("nan")
        o.fill_(float("nan"))
        torch.cuda.synchronize()
        assert api.gemm(prod, S, 3 * E, hidden, dx.data_ptr(), hidden, dw.data_ptr(), 3 * E, qkv[cached:].data_ptr(), ld, tile,
                        stream=s0.cuda_stream) == api.ERR.SUCCESS, api.last_error()
        assert L.cusync_hold_back(C.byref(prod.desc), s1.cuda_stream) == api.ERR.SUCCESS, api.last_error()
        assert api.attention(cons, S, heads, qkv.data_ptr(), ld, o.data_ptr(), E, cached_rows=cached, kv_split_blocks=blocks,
                             workspace=ws.data_ptr(), stream=s1.cuda_stream) == api.ERR.SUCCESS, api.last_error()
        torch.cuda.synchronize()
        prod.incrementIter()
        cons.incrementIter()
        full = np.ascontiguousarray(to_host(qkv)[:, :3 * E])
        assert np.array_equal(full[:cached].view(np.uint16), cache.view(np.uint16))
        assert_close(full[cached:], orc.gemm(x, w), "new rows")
        assert_close(to_host(o), orc.attention_kv(full, cached, heads, 128, True), "O")
    assert prod.read_state().spin_timeouts == 0 and cons.read_state().spin_timeouts == 0
    prod.destroy()
    cons.destroy()
