"""Convolutions under AvoidWaitKernel, whose caller has seen to it that all stages fit on the device at once: they stay with the
tiles' own kernels, whose workgroups cusync_conv2d_grid_split and cusync_conv2d_max_resident describe.  (Every pair that runs here
has fewer workgroups than the device has CUs, whichever kernel took it.)"""
import numpy as np
import pytest

import oracle as orc
from cusync_amd import _lib, api
from test_gpu_conv import he_filters, run_chain
from util import assert_close, empty_dev, to_dev, to_host, uniform_f16

pytestmark = pytest.mark.gpu

T128, T64 = api.CONV_TILE.HALO_128x128x64, api.CONV_TILE.HALO_64x128x64


# made and not run: few tiles in runs of steps, none in halves of columns
@pytest.mark.parametrize("shape,choice", [((1, 14, 14, 256), (T128, 4)), ((8, 28, 28, 128), (T128, 2)), ((11, 7, 7, 512), (T64, 7)), ((20, 14, 14, 256), (T128, 4))])
def test_choice(shape, choice):
    import torch
    N, H, W, Cc = shape
    dw = torch.zeros(Cc * 9 * Cc, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    for sync in (api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE):
        chain = api.ConvChain(N, H, W, Cc, [dw.data_ptr()] * 2, sync, opts=api.OPT.AVOID_WAIT_KERNEL)
        got = chain.tile(), chain.split()
        chain.destroy()
        assert got == choice, sync


def launched(chain, x, ys, layers):
    """Workgroups of each layer's launch in a run of the chain, from its timeline."""
    import torch
    L = _lib.load()
    buf = torch.zeros(1 + 8 * 4096, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    assert L.cusync_rt_set_timeline(buf.data_ptr(), buf.numel() * 8) == api.ERR.SUCCESS
    try:
        chain.run(x.data_ptr(), [y.data_ptr() for y in ys])
    finally:
        L.cusync_rt_set_timeline(None, 0)
    torch.cuda.synchronize()
    n = int(buf[0])
    rec = buf[1:1 + 8 * n].reshape(n, 8).cpu().numpy()
    role = rec[:, 0] & 255
    return [set(rec[role == r, 7].tolist()) for r in ((1, 2) if layers == 2 else (0,))]


def test_64_channels_stay_with_tiles():
    import torch
    N, H, W, Cc = 1, 56, 56, 64
    print("avoid wait, 64 channels", flush=True)
    dx, dws = to_dev(uniform_f16((N, H, W, Cc), 1)), [to_dev(he_filters(Cc, 3, 3, Cc, 2 + i)) for i in range(2)]
    dys = [empty_dev((N, H, W, Cc)) for _ in dws]
    torch.cuda.synchronize()
    for sync in (api.SYNC.ROW, api.SYNC.TILE):
        for opts, workgroups in ((-1, 49), (api.OPT.AVOID_WAIT_KERNEL, 13)):        # runs of 64 rows, tiles of 256
            chain = api.ConvChain(N, H, W, Cc, [w.data_ptr() for w in dws], sync, opts=opts)
            got = launched(chain, dx, dys, 2)
            chain.destroy()
            assert got == [{workgroups}] * 2, (sync, opts)


@pytest.mark.parametrize("shape", [(1, 56, 56, 64), (1, 14, 14, 256), (2, 7, 7, 512), (1, 28, 28, 128)])
def test_pairs(shape):
    print("avoid wait", shape, flush=True)
    outs = {}
    for sync in (api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE):
        x, ws, ys, states, _, _ = run_chain(*shape, 2, sync, runs=2, opts=api.OPT.AVOID_WAIT_KERNEL)
        assert all(st.spin_timeouts == 0 for st in states)
        outs[sync] = ys
    src = x
    for i in range(2):
        assert_close(outs[api.SYNC.STREAM][i], orc.conv2d_nhwc(src, ws[i], epilogue=orc.EPI_RELU if i == 0 else orc.EPI_NONE), "y%d" % i)
        src = outs[api.SYNC.STREAM][i]
        for sync in (api.SYNC.ROW, api.SYNC.TILE):
            assert np.array_equal(outs[sync][i].view(np.uint16), src.view(np.uint16)), (sync, i)


@pytest.mark.parametrize("tile,geom", [(T128, (2, 14, 14, 256, 256)), (T64, (1, 14, 14, 128, 128)), (T128, (1, 14, 14, 64, 128))])
@pytest.mark.parametrize("parts", [2, 4, 8])
def test_parts_of_a_tile_stay_runs(tile, geom, parts):
    """Bit for bit what the tile's own kernel gives, which a limit of one workgroup less than parts asks for as well."""
    import torch
    print("avoid wait parts", tile, geom, parts, flush=True)
    N, H, W, Cc, K = geom
    dx, dw = to_dev(uniform_f16((N, H, W, Cc), 3)), to_dev(he_filters(K, 3, 3, Cc, 4))
    grid = api.conv2d_grid(tile, N, H, W, K, 3, 3, 1, 1, parts)
    ws = torch.zeros(api.conv2d_workspace_size(N, H, W, Cc, K, tile, parts, 3, 3, 1, 1), dtype=torch.uint8, device="cuda")
    got = []
    for opts, limit in ((0, grid[0] * grid[1] * grid[2] - 1), (api.OPT.AVOID_WAIT_KERNEL, 0)):
        dy = empty_dev((N, H, W, K), fill=float("nan"))
        torch.cuda.synchronize()
        st = api.Stage(grid, (1, 1, 1), api.no_sync(), api.no_sync(), opts=opts)
        assert api.conv2d(st, N, H, W, Cc, K, dx.data_ptr(), dw.data_ptr(), dy.data_ptr(), tile, split_k=parts, max_workgroups=limit,
                          workspace=ws.data_ptr()) == api.ERR.SUCCESS, api.last_error()
        assert _lib.load().cusync_rt_device_sync() == 0, api.last_error()
        st.destroy()
        got.append(to_host(dy).view(np.uint16))
    assert np.array_equal(got[0], got[1])
