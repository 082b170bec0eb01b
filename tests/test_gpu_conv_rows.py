"""The convolution of 64 channels by rows (conv3x3_rows_kernel.h), which a chain runs by itself: images of one pixel, of one line and of
one column, rows that end inside a sixteen, inside a wavefront's turn and inside a tile, runs that cross tiles, one tile's rows
with several workgroups, against the CPU oracle.  Filters of small integers times a power of two and inputs of small integers keep
every sum exact (9 * 64 products of at most 4 each: below 2^24), so each layer's bits are the oracle's."""
import numpy as np
import pytest

import oracle as orc
from cusync_amd import api
from test_gpu_conv import run_chain
from util import assert_close, empty_dev, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 1, 300), (1, 300, 1), (2, 3, 3), (1, 5, 13), (1, 8, 8), (5, 7, 9), (1, 16, 16), (1, 17, 16), (7, 20, 21), (33, 1, 64),
                                   (3, 55, 57), (6, 56, 56), (32, 56, 56), (11, 24, 100)])
@pytest.mark.parametrize("sync", [api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE])
def test_chain_of_64_channels_exact(shape, sync):
    import torch
    print("conv rows", shape, sync, flush=True)
    N, H, W = shape
    rng = np.random.default_rng(N * H + W)
    xs = [rng.integers(-2, 3, (N, H, W, 64)).astype(np.float16) for _ in range(2)]
    ws = [rng.integers(-2, 3, (64, 3, 3, 64)).astype(np.float16), (rng.integers(-1, 2, (64, 3, 3, 64)) / 256).astype(np.float16)]
    dxs, dws = [to_dev(x) for x in xs], [to_dev(w) for w in ws]
    dys = [empty_dev((N, H, W, 64)) for _ in ws]
    torch.cuda.synchronize()
    chain = api.ConvChain(N, H, W, 64, [w.data_ptr() for w in dws], sync)
    assert (chain.tile(), chain.split()) == (api.CONV_TILE.HALO_256x64x64, 1)
    for dx in dxs:          # another image, the outputs full of NaN before each
        for y in dys:
            y.fill_(float("nan"))
        torch.cuda.synchronize()
        chain.run(dx.data_ptr(), [y.data_ptr() for y in dys])
    states = [chain.stage_state(i) for i in range(2)]
    chain.destroy()
    y1, y2 = (to_host(y) for y in dys)
    assert np.array_equal(y1.view(np.uint16), orc.conv2d_nhwc(xs[1], ws[0], epilogue=orc.EPI_RELU).view(np.uint16))
    # 576 products of sums up to 2304 with a quarter of a thousandth: fp32 has bits to spare
    assert np.array_equal(y2.view(np.uint16), orc.conv2d_nhwc(y1, ws[1]).view(np.uint16))
    for st in states:
        assert st.spin_timeouts == 0 and st.tile_counter == 0 and st.start_counter == 0
    if sync != api.SYNC.STREAM:
        assert states[0].kernel_executed == 2 and states[0].sems.size == -(-N * H * W // 256)
        d = states[0].desc
        p = orc.Policy(d.out.kind, d.out.order, d.out.tileM, d.out.tileN, d.out.waitValue, d.out.postValue, d.out.gridN, d.out.stride, d.out.R, d.out.S, d.out.H)
        assert np.array_equal(states[0].sems, orc.expected_sems_gemm(p, states[0].grid, 256, 64, 2, d.opts))


# 8 layers; an input tile with the filter too large for the LDS (the tile's own kernel runs)
@pytest.mark.parametrize("shape,layers", [((2, 30, 31), 8), ((2, 40, 300), 2), ((60, 56, 56), 2)])
def test_chain_of_64_channels(shape, layers):
    print("conv rows", shape, layers, flush=True)
    outs = {}
    for sync in (api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE):
        x, ws, ys, states, _, _ = run_chain(*shape, 64, layers, sync, runs=2)
        assert all(st.spin_timeouts == 0 for st in states)
        outs[sync] = ys
    src = x
    for i in range(layers):
        assert_close(outs[api.SYNC.STREAM][i], orc.conv2d_nhwc(src, ws[i], epilogue=orc.EPI_RELU if i + 1 < layers else orc.EPI_NONE), "y%d" % i)
        src = outs[api.SYNC.STREAM][i]
        for sync in (api.SYNC.ROW, api.SYNC.TILE):
            assert np.array_equal(outs[sync][i].view(np.uint16), src.view(np.uint16)), (sync, i)


def test_chain_of_64_channels_in_one_launch_or_with_a_tile_given():
    # what the caller fixes stays with the tile's own kernel; the sums differ in their order only
    N, H, W = 3, 28, 28
    x, ws, want, _, _, _ = run_chain(N, H, W, 64, 2, api.SYNC.ROW)
    for kw in (dict(fused=True), dict(tile=api.CONV_TILE.HALO_256x64x64), dict(tile=api.CONV_TILE.T128x64x32)):
        _, _, got, states, _, _ = run_chain(N, H, W, 64, 2, api.SYNC.ROW, **kw)
        assert all(st.spin_timeouts == 0 for st in states)
        for i in range(2):
            assert_close(got[i], want[i], "y%d" % i)


def test_overlapped_layers_leave_cus_free():
    # 20480 rows are 256 runs of 80; a consumer that finds no CU free is held back until its producer has started everywhere
    import torch
    from test_gpu_conv_avoid_wait import launched
    N, H, W = 5, 64, 64
    print("conv rows, CUs left", flush=True)
    rng = np.random.default_rng(3)
    dx = to_dev(rng.integers(-2, 3, (N, H, W, 64)).astype(np.float16))
    dws = [to_dev((rng.integers(-1, 2, (64, 3, 3, 64)) / 16).astype(np.float16)) for _ in range(2)]
    outs = []
    for sync, layers, workgroups in ((api.SYNC.STREAM, 1, 256), (api.SYNC.ROW, 2, 214), (api.SYNC.TILE, 2, 214)):
        dys = [empty_dev((N, H, W, 64), fill=float("nan")) for _ in range(layers)]
        torch.cuda.synchronize()
        chain = api.ConvChain(N, H, W, 64, [w.data_ptr() for w in dws[:layers]], sync, relu=False)
        assert launched(chain, dx, dys, layers) == [{workgroups}] * layers, sync
        chain.destroy()
        outs.append([to_host(y).view(np.uint16) for y in dys])
    assert np.array_equal(outs[1][0], outs[0][0]) and np.array_equal(outs[2][0], outs[0][0]) and np.array_equal(outs[1][1], outs[2][1])
