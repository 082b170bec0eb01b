"""cusync_conv2d_can_implement on the CPU (it launches nothing): an image so wide that the bytes of its halo wrap around 32 bits is
refused by the halo tiles, as every image that does not fit the LDS is."""
import ctypes as C

import pytest

from cusync_amd import _lib, api


@pytest.mark.parametrize("tile,W,Cc", [(api.CONV_TILE.HALO_256x64x64, (1 << 24) - 1, 64), (api.CONV_TILE.HALO_128x128x64, (1 << 23) - 1, 128),
                                       (api.CONV_TILE.HALO_64x128x64, (1 << 21) - 1, 512), (api.CONV_TILE.HALO_256x64x64, 1024, 64)])
def test_wide_images_are_refused(tile, W, Cc):
    L = _lib.load()
    a = _lib.Conv2dArgs()
    a.N, a.H, a.W, a.C, a.K, a.R, a.S, a.pad, a.stride = 1, 1, W, Cc, 8, 3, 3, 1, 1
    a.x = a.w = a.y = 4096
    a.tile, a.split_k = tile, 1
    a.stage.grid = L.cusync_conv2d_grid_split(tile, 1, 1, W, 8, 3, 3, 1, 1, 1)
    a.stage.tileOrder = a.stage.tileCounter = a.stage.startCounter = a.stage.spinTimeouts = a.stage.xcdTickets = 4096      # looked at, not read
    assert L.cusync_conv2d_can_implement(C.byref(a)) == api.ERR.NOT_INITIALIZED
    assert "halo" in api.last_error() or "LDS" in api.last_error()
