"""The kernels a few-row GEMM is dispatched to, at the edges of their ranges, exact on integer data."""
import ctypes as C

import numpy as np
import pytest

from cusync_amd import _lib, api
from util import empty_dev, to_dev, to_host

pytestmark = pytest.mark.gpu


def exact_gemm(tile, M, N, K, split_k):
    """A x B on small integers (every partial sum is exact in fp32 and fits fp16) against numpy; two launches on one
    workspace."""
    import torch
    L = _lib.load()
    rng = np.random.default_rng(1000 * tile + M)
    a = rng.integers(-2, 3, (M, K)).astype(np.float16)
    b = rng.integers(-2, 3, (K, N)).astype(np.float16)
    da, db, dd = to_dev(a), to_dev(b), empty_dev((M, N), fill=float("nan"))
    torch.cuda.synchronize()
    st = api.Stage(api.gemm_grid(tile, M, N, split_k), (1, 1, 1), api.no_sync(), api.no_sync())
    args = api.gemm_args(st, M, N, K, da.data_ptr(), K, db.data_ptr(), N, dd.data_ptr(), N, tile, split_k=split_k)
    ws = None
    if split_k > 1:
        ws = torch.zeros(L.cusync_gemm_workspace_size(C.byref(args)), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        args.workspace = ws.data_ptr()
    for _ in range(2):
        dd.fill_(float("nan"))
        torch.cuda.synchronize()
        assert L.cusync_gemm_run(C.byref(args), None) == api.ERR.SUCCESS, api.last_error()
        assert L.cusync_rt_device_sync() == 0, api.last_error()
        assert np.array_equal(to_host(dd), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float16))
    state = st.read_state()
    assert state.tile_counter == 0 and state.spin_timeouts == 0
    st.destroy()


@pytest.mark.parametrize("tile,rows", [(api.TILE.D32x128x64, 32), (api.TILE.D64x128x64, 64), (api.TILE.D64x192x64, 64)])
@pytest.mark.parametrize("more", [-1, 0, 1])
@pytest.mark.parametrize("split_k", [1, 3])
def test_one_row_tile_and_the_next(tile, rows, more, split_k):
    # up to `rows` rows the weights are read by one row tile (non-temporal loads), one row more and by two
    print("few rows", tile, rows + more, split_k, flush=True)
    exact_gemm(tile, rows + more, 328, 520, split_k)


@pytest.mark.parametrize("tile", [api.TILE.D32x128x64, api.TILE.D64x128x64, api.TILE.D64x192x64])
@pytest.mark.parametrize("K", [8, 64, 72, 200, 320, 392, 456])
def test_fewer_chunks_than_stages(tile, K):
    # the prologue sends out all of B's first chunks ahead of A's: one chunk of K, as many as the pipeline has stages, one more
    print("few chunks", tile, K, flush=True)
    exact_gemm(tile, 20, 328, K, 1)


@pytest.mark.parametrize("policy_kind", ["row", "tile"])
@pytest.mark.parametrize("tile", [api.TILE.D32x128x64, api.TILE.D64x128x64, api.TILE.D64x192x64])
@pytest.mark.parametrize("K,N1,N2,split2", [(72, 328, 1992, 1), (72, 328, 33288, 1), (520, 1416, 4104, 2), (328, 2568, 520, 3), (200, 1536, 3584, 2), (72, 3080, 520, 1)])
def test_one_row_of_tiles_in_one_launch(policy_kind, tile, K, N1, N2, split2):
    # two GEMMs of one row of tiles in one launch: the second one's lists begin a position further on (K = 200, whose weights'
    # rows are multiples of 1 KiB apart), its weights are fetched, under ReorderTileLoads before the first one's tiles are waited for (not with more
    # tiles than CUs, nor under a tile policy with N1 = 3080); lists of unequal length, N and K not multiples of the tile
    import torch
    L = _lib.load()
    rows = api.tile_shape(tile)[0]
    # (limit: workgroups that work through several tiles of each GEMM, most of them drawn)
    for M, opts, limit in ((1, api.OPT.REORDER_TILE_LOADS, 0), (rows, api.OPT.REORDER_TILE_LOADS, 0), (rows, 0, 0), (rows, api.OPT.REORDER_TILE_LOADS, 3)):
        print("one launch", policy_kind, tile, M, K, N1, N2, split2, opts, limit, flush=True)
        rng = np.random.default_rng(tile + M + K)
        a, b = rng.integers(-1, 2, (M, K)).astype(np.float16), rng.integers(-1, 2, (K, N1)).astype(np.float16)
        d = rng.integers(-1, 2, (N1, N2)).astype(np.float16)
        da, db, dd = to_dev(a), to_dev(b), to_dev(d)
        dc, de = empty_dev((M, N1), fill=float("nan")), empty_dev((M, N2), fill=float("nan"))
        grids = [api.gemm_grid(tile, M, N1, 1), api.gemm_grid(tile, M, N2, split2)]
        tm, tn, _ = api.tile_shape(tile)
        pol = api.tile_sync(api.ORDER.TRANSPOSE_XY, tm, tn) if policy_kind == "tile" else api.row_sync(tm, grids[0][0])
        st = [api.Stage(grids[0], (1, 1, 1), api.no_sync(), pol, opts=opts), api.Stage(grids[1], (1, 1, 1), pol, api.no_sync(), opts=opts)]
        assert api.set_producer_consumer_pair(st[0], st[1]) == api.ERR.SUCCESS
        args = (_lib.GemmArgs * 2)(
            api.gemm_args(st[0], M, N1, K, da.data_ptr(), K, db.data_ptr(), N1, dc.data_ptr(), N1, tile, max_workgroups=limit),
            api.gemm_args(st[1], M, N2, N1, dc.data_ptr(), N1, dd.data_ptr(), N2, de.data_ptr(), N2, tile, split_k=split2))
        ws = None
        if split2 > 1:
            ws = torch.zeros(L.cusync_gemm_workspace_size(C.byref(args[1])), dtype=torch.uint8, device="cuda")
            args[1].workspace = ws.data_ptr()
        c = a.astype(np.float64) @ b.astype(np.float64)
        assert np.abs(c).max() < 2048          # exact in fp16
        e = (c @ d.astype(np.float64)).astype(np.float16)
        for it in range(3):
            for t in (dc, de):
                t.fill_(float("nan"))
            torch.cuda.synchronize()
            assert L.cusync_gemm_chain_run(args, 2, None) == api.ERR.SUCCESS, api.last_error()
            assert L.cusync_rt_device_sync() == 0, api.last_error()
            for k in range(2):
                st[k].incrementIter()
                args[k].stage = st[k].desc
            assert np.array_equal(to_host(dc), c.astype(np.float16)) and np.array_equal(to_host(de), e), it
        states = [s_.read_state() for s_ in st]
        for s_ in st:
            s_.destroy()
        assert all(s_.spin_timeouts == 0 and s_.tile_counter == 0 for s_ in states)


@pytest.mark.parametrize("policy_kind", ["row", "tile"])
@pytest.mark.parametrize("tile", [api.TILE.D32x128x64, api.TILE.D64x128x64, api.TILE.D64x192x64])
def test_weights_written_ahead_of_the_producer_on_its_stream(policy_kind, tile):
    # a consumer under AvoidWaitKernel and without ReorderTileLoads reaches the device before its producer; its weights are
    # written on the producer's stream, ahead of the producer: the wait for the producer's tiles is what orders them.  (The
    # producer's stream is filled first: two streams may share a hardware queue, and the consumer must not be in front there.)
    import torch
    print("weights behind the wait", policy_kind, tile, flush=True)
    M, K, N1, N2 = 20, 64, 512, 512
    rng = np.random.default_rng(tile)
    a, b = rng.integers(-1, 2, (M, K)).astype(np.float16), rng.integers(-1, 2, (K, N1)).astype(np.float16)
    d = rng.integers(-1, 2, (N1, N2)).astype(np.float16)
    da, db, src = to_dev(a), to_dev(b), to_dev(d)
    w, c, e = empty_dev((N1, N2), fill=0.0), empty_dev((M, N1), fill=float("nan")), empty_dev((M, N2), fill=float("nan"))
    filler = torch.zeros(64 << 20, device="cuda")
    tm, tn, _ = api.tile_shape(tile)
    g1, g2 = api.gemm_grid(tile, M, N1), api.gemm_grid(tile, M, N2)
    pol = api.tile_sync(api.ORDER.TRANSPOSE_XY, tm, tn) if policy_kind == "tile" else api.row_sync(tm, g1[0])
    prod = api.Stage(g1, (1, 1, 1), api.no_sync(), pol, opts=api.OPT.AVOID_WAIT_KERNEL)
    cons = api.Stage(g2, (1, 1, 1), pol, api.no_sync(), opts=api.OPT.AVOID_WAIT_KERNEL)
    assert api.set_producer_consumer_pair(prod, cons) == api.ERR.SUCCESS
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        for _ in range(24):                   # two milliseconds and more in which the consumer gets to the device and waits
            filler.add_(1)
        w.add_(src)
    assert api.gemm(prod, M, N1, K, da.data_ptr(), K, db.data_ptr(), N1, c.data_ptr(), N1, tile, stream=first.cuda_stream) == api.ERR.SUCCESS, api.last_error()
    assert api.gemm(cons, M, N2, N1, c.data_ptr(), N1, w.data_ptr(), N2, e.data_ptr(), N2, tile, stream=second.cuda_stream) == api.ERR.SUCCESS, api.last_error()
    torch.cuda.synchronize()
    ps, cs = prod.read_state(), cons.read_state()
    prod.destroy(); cons.destroy()
    assert ps.spin_timeouts == 0 and cs.spin_timeouts == 0
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(want).max() < 2048
    assert np.array_equal(to_host(e), (want @ d.astype(np.float64)).astype(np.float16))
