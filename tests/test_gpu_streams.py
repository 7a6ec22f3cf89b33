"""Calls on GPU frames that the caller's stream is still computing: every entry
point starts after the work queued on the device's default stream, and the
Python ones after that of torch's current stream.

The frames are written behind some tens of ms of matrix products; the call
comes while these run, and its rows are those of a call after a
synchronisation, bit for bit."""
import ctypes

import numpy as np
import pytest

from tracking_optimizations_amd import _lib
from tracking_optimizations_amd._lib import GT_FRAMES_ON_DEVICE, Adjoint, Result, check, load
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu

N, H, W = 2, 200, 240
PARAMS = dict(diameter=7, separation=8, minmass=100)


def _frames(seed):
    rng = np.random.default_rng(seed)
    yy, xx = np.mgrid[:H, :W]
    f = rng.poisson(60, (N, H, W)).astype(np.float64)
    for k in range(60):
        y, x, a = rng.uniform(0, H), rng.uniform(0, W), rng.uniform(200, 900)
        f[k % N] += a * np.exp(-((yy - y) ** 2 + (xx - x) ** 2) / (2 * 1.6 ** 2))
    return f.astype(np.int16)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _c_locate(dtype):
    def call(ctx, video, p):
        out = ctypes.c_void_p()
        fn = load().gt_locate_u16 if dtype == "u16" else load().gt_locate_f32
        check(fn(ctx.handle, _ptr(video), N, H, W, ctypes.byref(p), GT_FRAMES_ON_DEVICE,
                 ctypes.byref(out)))
        return Result(out).rows()
    return call


def _c_batch(ctx, video, p):
    out = ctypes.c_void_p()
    desc = (_lib.GtFrameDesc * N)()
    for i in range(N):
        desc[i].data, desc[i].h, desc[i].w, desc[i].frame_index = video[i].data_ptr(), H, W, i
    check(load().gt_locate_batch(ctx.handle, desc, N, 0, ctypes.byref(p), GT_FRAMES_ON_DEVICE,
                                 ctypes.byref(out)))
    return Result(out).rows()


def _c_adjoint(ctx, video, p):
    out = ctypes.c_void_p()
    check(load().gt_locate_adjoint(ctx.handle, _ptr(video), 0, N, H, W, ctypes.byref(p),
                                   GT_FRAMES_ON_DEVICE, ctypes.byref(out)))
    a = Adjoint(out, N, H, W)
    return np.concatenate([a.rows(), a.sigma()], axis=1)


def _errors(ctx, video, p):
    from tracking_optimizations_amd.adjoint import locate_errors
    rows, _cand, sigma, _a = locate_errors(video, p, ctx=ctx)
    return np.concatenate([rows, sigma], axis=1)


def _locate(ctx, video, p):
    return locate(video, p, ctx=ctx)[0]


CALLS = {"gt_locate_u16": (_c_locate("u16"), "u16"), "gt_locate_f32": (_c_locate("f32"), "f32"),
         "gt_locate_batch": (_c_batch, "u16"), "gt_locate_adjoint": (_c_adjoint, "u16"),
         "locate": (_locate, "u16"), "locate_errors": (_errors, "u16")}


# C callers are ordered after the default stream only
@pytest.mark.parametrize("name,side", [(n, False) for n in sorted(CALLS)] +
                         [("locate", True), ("locate_errors", True)])
@pytest.mark.parametrize("graphs", [False, True])
def test_frames_still_being_computed(name, side, graphs):
    torch = pytest.importorskip("torch")
    torch.cuda.init()   # before the first context of a process
    call, dtype = CALLS[name]
    # streams share hardware queues, and two on one queue run in order by
    # themselves: the streams of several contexts are on all of them
    ctxs = [_lib.Context(0) for _ in range(4)]
    p = make_params(**PARAMS)
    src = [torch.from_numpy(_frames(s)).cuda() for s in (1, 2)]
    if dtype == "f32":
        src = [s.float() for s in src]
    video = torch.zeros_like(src[0])
    view = video.view(torch.uint16) if dtype == "u16" else video
    ref = []
    for s in src:
        video.copy_(s)
        torch.cuda.synchronize()
        ref.append(call(ctxs[0], view, p))
    assert len(ref[0]) > 10 and not np.array_equal(ref[0], ref[1])
    for ctx in ctxs:   # buffers, and where asked for the graph
        ctx.set_graphs(graphs)
        np.testing.assert_array_equal(call(ctx, view, p), ref[1])
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    with torch.cuda.stream(stream):
        m = torch.randn(4096, 4096, device="cuda")
        for q, ctx in zip((0, 1, 0, 1), ctxs):
            stream.synchronize()
            for _ in range(20):
                m = (m @ m).clamp_(-1, 1)
            video.copy_(src[q])
            assert not stream.query()   # the frames are not there yet
            got = call(ctx, view, p)
            np.testing.assert_array_equal(got, ref[q])


def test_device_rows_still_being_read():
    """Rows left on the GPU, copied on the default stream behind other work:
    the next call on the context does not overwrite them before that."""
    torch = pytest.importorskip("torch")
    torch.cuda.init()
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpyAsync.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int,
                                   ctypes.c_void_p]
    p = make_params(**PARAMS)
    first, second = _frames(1).view(np.uint16), _frames(2).view(np.uint16)
    video = torch.from_numpy(_frames(1)).cuda()
    m = torch.randn(4096, 4096, device="cuda")
    for ctx in [_lib.Context(0) for _ in range(4)]:
        ref = locate(first, p, ctx=ctx)[0]
        locate(second, p, ctx=ctx)
        out = ctypes.c_void_p()
        check(load().gt_locate_u16(ctx.handle, _ptr(video), N, H, W, ctypes.byref(p),
                                   GT_FRAMES_ON_DEVICE | _lib.GT_RESULT_ON_DEVICE, ctypes.byref(out)))
        res = Result(out)
        rows = torch.zeros(ref.shape, device="cuda")
        torch.cuda.synchronize()
        for _ in range(20):
            m = (m @ m).clamp_(-1, 1)
        assert hip.hipMemcpyAsync(rows.data_ptr(), res.device_ptr(), ref.nbytes, 3, None) == 0
        locate(second, p, ctx=ctx)
        np.testing.assert_array_equal(rows.cpu().numpy(), ref)
