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
