"""The chain handles return when their outputs are in memory, on the word of the device's own stamps."""
import time

import numpy as np
import pytest

from cusync_amd import api
from util import empty_dev, normal_f16, to_dev, uniform_f16

pytestmark = pytest.mark.gpu


def chain(kind, sync):
    """(handle, one pass as a call that returns its times, the buffers a pass fills)"""
    if kind == "conv":
        N, H, C = 8, 28, 128
        x = to_dev(uniform_f16((N, H, H, C), 1))
        ws = [to_dev(normal_f16((C, 3, 3, C), k, std=0.03)) for k in (2, 3, 4)]
        ys = [empty_dev((N, H, H, C)) for _ in ws]
        h = api.ConvChain(N, H, H, C, [w.data_ptr() for w in ws], sync)
        return h, lambda: h.run(x.data_ptr(), [y.data_ptr() for y in ys]), ys + [x] + ws, len(ys)
    if kind in ("attention", "attention of few rows"):
        S, cached, hidden, heads = 40 if kind == "attention" else 17, 300, 1024, 3
        E = heads * 128
        x, wqkv, wo = to_dev(uniform_f16((S, hidden), 1)), to_dev(normal_f16((hidden, 3 * E), 2)), to_dev(normal_f16((E, hidden), 3))
        qkv, o, y = to_dev(normal_f16((cached + S, 3 * E), 4, std=1.0)), empty_dev((S, E)), empty_dev((S, hidden))
        h = api.AttnLayer(S, hidden, heads, sync, wqkv.data_ptr(), wo.data_ptr(), cached_rows=cached)
        return h, lambda: h.run(x.data_ptr(), qkv.data_ptr(), o.data_ptr(), y.data_ptr()), [o, y, qkv, x, wqkv, wo], 2
    model, rows, one, where = kind
    hidden, inner = 4096, 2816
    n1 = inner * (2 if model == api.MODEL.LLAMA else 1)
    x, w1, w2 = to_dev(uniform_f16((rows, hidden), 1)), to_dev(normal_f16((hidden, n1), 2)), to_dev(normal_f16((inner, hidden), 3))
    hb, y = empty_dev((rows, inner if where == 0 else n1)), empty_dev((rows, hidden))
    h = api.Mlp(model, rows, hidden, inner, sync, w1.data_ptr(), w2.data_ptr(), one_launch=one, swiglu_in_gemm2=where)
    return h, lambda: h.run(x.data_ptr(), hb.data_ptr(), y.data_ptr()), [hb, y, x, w1, w2], 2


@pytest.mark.parametrize("sync", [api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE])
@pytest.mark.parametrize("kind", [(api.MODEL.GPT3, 1, -1, 0), (api.MODEL.GPT3, 40, 0, 0), (api.MODEL.GPT3, 700, -1, 0), (api.MODEL.LLAMA, 300, -1, 0),
                                  (api.MODEL.LLAMA, 300, -1, -1), (api.MODEL.LLAMA, 300, -1, 1), "conv", "attention",
                                  "attention of few rows"])
def test_outputs_are_there_when_a_run_returns(kind, sync):
    import torch
    print("run returns", kind, sync, flush=True)
    torch.cuda.synchronize()
    handle, run, buffers, outputs = chain(kind, sync)
    copies = [torch.empty_like(b) for b in buffers[:outputs]]
    other = torch.cuda.Stream()
    for _ in range(20):
        for b in buffers[:outputs]:
            b.fill_(float("nan"))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        (us,) = run()
        wall = (time.perf_counter() - t0) * 1e6
        with torch.cuda.stream(other):            # a stream that knows nothing of the chain's
            for c, b in zip(copies, buffers):
                c.copy_(b, non_blocking=True)
        torch.cuda.synchronize()
        assert 0 < us < wall
        for c, b in zip(copies, buffers):
            assert torch.equal(c.view(torch.int16), b.view(torch.int16))
            assert not torch.isnan(b).any()
    handle.destroy()


@pytest.mark.parametrize("sync", [api.SYNC.STREAM, api.SYNC.ROW])
@pytest.mark.parametrize("kind", [(api.MODEL.GPT3, 1, -1, 0), (api.MODEL.GPT3, 700, -1, 0), "conv", "attention"])
def test_diagnosis_records_are_there_when_a_run_returns(kind, sync):
    import torch
    from cusync_amd import _lib
    print("records", kind, sync, flush=True)
    L = _lib.load()
    torch.cuda.synchronize()
    handle, run, b, outputs = chain(kind, sync)
    # (attention: not the third stage, whose 64x128x64 tile is register-staged and keeps no records)
    tiles = sum(int(np.prod(handle.stage_state(i).grid)) for i in range(outputs))
    other = torch.cuda.Stream()
    try:
        for _ in range(10):
            buf = torch.zeros(1 + 8 * (tiles + 8), dtype=torch.int64, device="cuda")
            early = torch.empty_like(buf)
            torch.cuda.synchronize()
            assert L.cusync_rt_set_timeline(buf.data_ptr(), buf.numel() * 8) == api.ERR.SUCCESS
            run()
            with torch.cuda.stream(other):        # a stream that knows nothing of the chain's
                early.copy_(buf, non_blocking=True)
            other.synchronize()
            L.cusync_rt_set_timeline(None, 0)
            torch.cuda.synchronize()
            assert torch.equal(early, buf)
            r = buf.cpu().numpy()
            assert r[0] == tiles
            rec = r[1:1 + 8 * tiles].reshape(-1, 8)
            assert (rec[:, 2:] > 0).all() and (rec[:, 5] >= rec[:, 2]).all()
    finally:
        L.cusync_rt_set_timeline(None, 0)
    torch.cuda.synchronize()
    handle.destroy()


@pytest.mark.parametrize("sync", [api.SYNC.STREAM, api.SYNC.ROW, api.SYNC.TILE])
@pytest.mark.parametrize("kind", [(api.MODEL.GPT3, 1, -1, 0), (api.MODEL.GPT3, 40, 0, 0), (api.MODEL.LLAMA, 300, -1, -1), "conv", "attention"])
def test_a_refused_run_has_launched_nothing(kind, sync):
    """A last output that is not aligned is found before the stages in front of it are launched: the outputs stay as they
    were, and the next run counts its stages from where the last whole run left them."""
    import torch
    print("run refused", kind, sync, flush=True)
    torch.cuda.synchronize()
    handle, run, b, outputs = chain(kind, sync)
    p = [t.data_ptr() for t in b]
    if kind == "conv":
        refused = lambda: handle.run(p[outputs], p[:outputs - 1] + [p[outputs - 1] + 2])
    elif kind == "attention":
        refused = lambda: handle.run(p[3], p[2], p[0], p[1] + 2)
    else:
        refused = lambda: handle.run(p[2], p[0], p[1] + 2)
    run()
    torch.cuda.synchronize()
    want = [t.clone() for t in b[:outputs]]
    for _ in range(3):
        for t in b[:outputs]:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        with pytest.raises(api.CuSyncError):
            refused()
        torch.cuda.synchronize()
        assert all(bool(torch.isnan(t).all()) for t in b[:outputs])
        run()
        torch.cuda.synchronize()
        for t, w in zip(b, want):
            assert torch.equal(t.view(torch.int16), w.view(torch.int16))
    handle.destroy()


def test_split_times_add_up():
    import torch
    torch.cuda.synchronize()
    rows, hidden, inner = 64, 4096, 2816
    x, w1, w2 = to_dev(uniform_f16((rows, hidden), 1)), to_dev(normal_f16((hidden, inner), 2)), to_dev(normal_f16((inner, hidden), 3))
    h, y = empty_dev((rows, inner)), empty_dev((rows, hidden))
    torch.cuda.synchronize()
    m = api.Mlp(api.MODEL.GPT3, rows, hidden, inner, api.SYNC.STREAM, w1.data_ptr(), w2.data_ptr())
    total, g1, g2 = m.run(x.data_ptr(), h.data_ptr(), y.data_ptr(), runs=5, split=True)
    m.destroy()
    assert np.allclose(np.array(g1) + np.array(g2), total, atol=0.02) and min(g1) > 0 and min(g2) > 0


def run_two_at_once(handles, bufs):
    """50 passes of each handle from a host thread of its own; every output is what the handle gave alone."""
    import threading
    import torch
    alone, failed = [], []
    for h, (x, mid, y) in zip(handles, bufs):
        h.run(x.data_ptr(), mid.data_ptr(), y.data_ptr())
        alone.append(y.clone())
        y.fill_(float("nan"))
    torch.cuda.synchronize()

    def work(h, x, mid, y):
        try:
            for _ in range(50):
                h.run(x.data_ptr(), mid.data_ptr(), y.data_ptr())
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(h,) + b) for h, b in zip(handles, bufs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for (x, mid, y), want, h in zip(bufs, alone, handles):
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        h.destroy()


def test_two_launches_of_several_gemms_at_once():
    # both GEMMs of a handle in one launch whose workgroups wait for each other; 64x128 tiles leave a CU to two workgroups in
    # every kernel, and two times 240 fit the device
    import torch
    from cusync_amd import _lib
    print("two launches at once", flush=True)
    L = _lib.load()
    assert [L.cusync_gemm_max_resident(t) // L.cusync_gemm_max_resident(api.TILE.T256x192x64) for t in
            (api.TILE.D32x128x64, api.TILE.D64x128x64, api.TILE.D64x192x64)] == [1, 2, 1]
    hidden, inner, rows = 12288, 6144, 64
    w1, w2 = to_dev(normal_f16((hidden, inner), 2, std=0.02)), to_dev(normal_f16((inner, hidden), 3, std=0.02))
    bufs = [(to_dev(uniform_f16((rows, hidden), 4 + k)), empty_dev((rows, inner)), empty_dev((rows, hidden))) for k in range(2)]
    torch.cuda.synchronize()
    tile = api.TILE.D64x128x64
    handles = [api.Mlp(api.MODEL.GPT3, rows, hidden, inner, api.SYNC.ROW, w1.data_ptr(), w2.data_ptr(), tile1=tile, tile2=tile, one_launch=True) for _ in bufs]
    assert all(int(np.prod(h.stage_state(0).grid)) <= L.cusync_gemm_max_resident(tile) // 2 for h in handles)
    run_two_at_once(handles, bufs)


@pytest.mark.parametrize("rows", [300, 512])
def test_two_launches_whose_slices_wait_for_each_other_at_once(rows):
    # GEMM1 of a LLaMA MLP, 174 or 232 workgroups to a handle on 256 CUs: each handle's slices may hold the CUs the other's
    # siblings need, and then give their tiles up
    import torch
    print("two launches of slices at once", rows, flush=True)
    hidden, inner = 8192, 2752
    w1, w2 = to_dev(normal_f16((hidden, 2 * inner), 2, std=0.02)), to_dev(normal_f16((inner, hidden), 3, std=0.02))
    bufs = [(to_dev(uniform_f16((rows, hidden), 4 + k)), empty_dev((rows, inner)), empty_dev((rows, hidden))) for k in range(2)]
    torch.cuda.synchronize()
    handles = [api.Mlp(api.MODEL.LLAMA, rows, hidden, inner, api.SYNC.ROW, w1.data_ptr(), w2.data_ptr()) for _ in bufs]
    assert handles[0].splits()[0] > 1
    run_two_at_once(handles, bufs)
