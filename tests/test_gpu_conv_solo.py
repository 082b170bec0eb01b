"""The convolution kernel whose wavefronts each take whole units of the sum (conv3x3_solo_kernel.h), at the edges of its tiles,
columns and runs, against the CPU oracle: with small integers every order of adding is exact (at most 9 * 512 * 4 < 2^24), and the
oracle rounds to halfs as the kernel does."""
import numpy as np
import pytest

import oracle as orc
from cusync_amd import api
from test_gpu_conv import he_filters, run_chain, run_conv
from util import assert_close, uniform_f16

pytestmark = pytest.mark.gpu

T128, T64 = api.CONV_TILE.HALO_128x128x64, api.CONV_TILE.HALO_64x128x64


def integers(geom, seed):
    N, H, W, Cc, K = geom
    rng = np.random.default_rng(seed)
    return rng.integers(-2, 3, (N, H, W, Cc)).astype(np.float16), rng.integers(-2, 3, (K, 3, 3, Cc)).astype(np.float16)


# one pixel; a row more and a row less than a tile; a lone column of images; columns in one half only, just in both, ragged;
# 64 channels (nine units for four wavefronts), 512 (the halo that just fits)
@pytest.mark.parametrize("tile,geom", [(T128, (1, 1, 1, 128, 8)), (T128, (1, 129, 1, 256, 64)), (T128, (1, 1, 127, 128, 72)), (T128, (3, 14, 14, 256, 136)),
                                       (T128, (2, 12, 12, 64, 264)), (T64, (1, 65, 1, 128, 128)), (T64, (3, 7, 7, 512, 264)), (T64, (1, 3, 21, 64, 72)),
                                       (T64, (2, 9, 13, 256, 200))])
@pytest.mark.parametrize("parts", [2, 4, 8])
def test_parts_of_a_tile(tile, geom, parts):
    print("conv parts", tile, geom, parts, flush=True)
    x, w = integers(geom, geom[3] + geom[4])
    got = run_conv(x, w, tile, launches=2, split_k=parts, epilogue=api.EPI.RELU)
    assert np.array_equal(got.view(np.uint16), orc.conv2d_nhwc(x, w, epilogue=orc.EPI_RELU).view(np.uint16))


def test_fewer_workgroups_than_parts_take_the_tile_in_runs():
    # the kernel needs a workgroup per part: under a limit, and where the parts are more than stay resident, the other one runs
    print("conv parts, limited", flush=True)
    x, w = integers((2, 14, 14, 256, 256), 1)
    want = orc.conv2d_nhwc(x, w).view(np.uint16)
    for limit in (0, 15, 16, 3):
        assert np.array_equal(run_conv(x, w, T128, split_k=2, max_workgroups=limit).view(np.uint16), want), limit
    x, w = integers((21, 14, 14, 128, 256), 2)          # 65 * 2 * 2 = 260 parts of 64-row tiles
    assert np.array_equal(run_conv(x, w, T64, split_k=2).view(np.uint16), orc.conv2d_nhwc(x, w).view(np.uint16))


# the built-in choice on both sides of its lines: 64-row tiles in halves, 128-row tiles in halves, neither; 512 channels in four runs a
# half, in two, in none
@pytest.mark.parametrize("shape,choice", [((20, 14, 14, 256), (T64, 2)), ((21, 14, 14, 256), (T128, 2)), ((10, 28, 28, 128), (T64, 2)), ((20, 28, 28, 128), (T128, 2)),
                                          ((21, 28, 28, 128), (T128, 1)), ((10, 7, 7, 512), (T64, 8)), ((11, 7, 7, 512), (T64, 4)), ((21, 7, 7, 512), (T64, 2))])
def test_chain_choice(shape, choice):
    print("conv chain choice", shape, flush=True)
    outs = {}
    for sync in (api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE):
        x, ws, ys, states, tile, _ = run_chain(*shape, 3, sync, runs=2)
        assert (tile, run_chain.split) == choice
        assert all(st.spin_timeouts == 0 for st in states)
        outs[sync] = ys
    src = x
    for i in range(3):
        assert_close(outs[api.SYNC.STREAM][i], orc.conv2d_nhwc(src, ws[i], epilogue=orc.EPI_RELU if i < 2 else orc.EPI_NONE), "y%d" % i)
        src = outs[api.SYNC.STREAM][i]
        for sync in (api.SYNC.ROW, api.SYNC.TILE):
            assert np.array_equal(outs[sync][i].view(np.uint16), src.view(np.uint16)), (sync, i)


def test_chain_whose_halo_leaves_no_room_for_halves():
    # 512 channels, 16 wide: the halo fits beside the 48 KB ring of the tile's own kernel and not beside 64 KB; its tiles take eight runs
    print("conv chain in runs", flush=True)
    outs = {}
    for sync in (api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE):
        x, ws, ys, states, tile, _ = run_chain(1, 16, 16, 512, 2, sync, runs=2)
        assert (tile, run_chain.split) == (T64, 8)
        assert all(st.spin_timeouts == 0 for st in states)
        outs[sync] = ys
    for i, src in enumerate((x, outs[api.SYNC.STREAM][0])):
        assert_close(outs[api.SYNC.STREAM][i], orc.conv2d_nhwc(src, ws[i], epilogue=orc.EPI_RELU if i == 0 else orc.EPI_NONE), "y%d" % i)
        for sync in (api.SYNC.ROW, api.SYNC.TILE):
            assert np.array_equal(outs[sync][i].view(np.uint16), outs[api.SYNC.STREAM][i].view(np.uint16)), (sync, i)


def test_rounding_of_parts():
    # random operands: the distance the other tiles' tests allow
    for tile, parts in ((T128, 2), (T128, 4), (T64, 8)):
        x, w = uniform_f16((2, 14, 14, 256), 21), he_filters(256, 3, 3, 256, 22)
        assert_close(run_conv(x, w, tile, split_k=parts), orc.conv2d_nhwc(x, w), "y")


def test_chain_allocates_what_it_adds_up():
    # two halves of columns share a tile and add nothing up through memory: 16 layers of 20x14x14x256, 124 tiles of 64x128 each, had
    # 130 MB of partial sums between them; 64 channels have a word per tile.  (What else a handle holds is far below this line.)
    import torch
    for shape, choice in (((20, 14, 14, 256), (T64, 2)), ((32, 56, 56, 64), (api.CONV_TILE.HALO_256x64x64, 1))):
        Cc = shape[3]
        dw = torch.zeros(Cc * 9 * Cc, dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        chain = api.ConvChain(*shape, [dw.data_ptr()] * 16, api.SYNC.STREAM)
        taken = free - torch.cuda.mem_get_info()[0]
        got = chain.tile(), chain.split()
        chain.destroy()
        assert got == choice and taken < 48 << 20, (shape, taken)
