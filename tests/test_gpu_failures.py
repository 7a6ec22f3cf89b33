"""Allocation failures forced from the host (gt_debug_inject_alloc_failure):
the call returns GT_E_OOM instead of aborting (the reference panics,
execute_gpu.rs:497-499, gpu_setup.rs:201,208), the context keeps working,
and the next call gives the rows of an untouched context."""
import ctypes

import numpy as np
import pytest

from tracking_optimizations_amd import _lib, synth
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu

KW = dict(diameter=9, minmass=1000, separation=9, percentile=64)


@pytest.fixture(scope="module")
def frames():
    return synth.generate_host(_lib.default_context(0), synth.single_512(seed=1, n_frames=2))


@pytest.fixture(scope="module")
def reference(frames):
    return locate(frames, make_params(**KW), ctx=_lib.Context(0))


def _inject(kind, after):
    _lib.check(_lib.load().gt_debug_inject_alloc_failure(kind, after))


@pytest.mark.parametrize("after", [1, 2, 4, 7, 10])
def test_device_allocation_failure(frames, reference, after):
    ctx = _lib.Context(0)           # fresh: its first call allocates its workspaces
    _inject(0, after)
    try:
        with pytest.raises(_lib.GtError) as e:
            locate(frames, make_params(**KW), ctx=ctx)
    finally:
        _inject(0, 0)
    assert e.value.status == _lib.GT_E_OOM, str(e.value)
    print(f"[failure] device allocation {after}: {e.value}", flush=True)
    got = locate(frames, make_params(**KW), ctx=ctx)
    assert np.array_equal(got[0], reference[0]) and np.array_equal(got[1], reference[1])


def test_host_allocation_failure(frames, reference):
    ctx = _lib.Context(0)
    _inject(1, 1)
    try:
        with pytest.raises(_lib.GtError) as e:
            locate(frames, make_params(**KW), ctx=ctx)
    finally:
        _inject(1, 0)
    assert e.value.status == _lib.GT_E_OOM, str(e.value)
    got = locate(frames, make_params(**KW), ctx=ctx)
    assert np.array_equal(got[0], reference[0]) and np.array_equal(got[1], reference[1])


def test_pinned_staging_failure(reference):
    """Host frames of a movie of several pinned chunks: the pinned staging
    buffers cannot be had; then they can."""
    ctx = _lib.Context(0)
    big = synth.generate_host(ctx, synth.movie_2048(seed=2, n_frames=34))
    p = make_params(diameter=11, separation=11, smoothing_size=11, percentile=64)
    ref = locate(big, p, ctx=_lib.Context(0))
    for after in (1, 2):
        c = _lib.Context(0)
        _inject(0, after)
        try:
            with pytest.raises(_lib.GtError) as e:
                locate(big, p, ctx=c)
        finally:
            _inject(0, 0)
        assert e.value.status == _lib.GT_E_OOM
        got = locate(big, p, ctx=c)
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])


def test_disarmed_by_zero(frames, reference):
    _inject(0, 3)
    _inject(0, 0)
    got = locate(frames, make_params(**KW), ctx=_lib.Context(0))
    assert np.array_equal(got[0], reference[0])
    with pytest.raises(_lib.GtError):
        _inject(2, 1)


@pytest.mark.parametrize("kind", [0, 1])
def test_adjoint_allocation_failures(frames, kind):
    """Each allocation of an adjoint in turn, on the device (workspaces, rows,
    patches, the frames' row ranges) and for its host results: GT_E_OOM, and
    the next call's rows, errors and patches are an untouched context's."""
    from tracking_optimizations_amd.adjoint import _adjoint
    p = make_params(**KW)
    want = _adjoint(frames, p, True, ctx=_lib.Context(0))
    want = [want.rows(), want.sigma(), want.origin(), want.jacobian()]
    failed = 0
    for after in range(1, 25):
        ctx = _lib.Context(0)
        _inject(kind, after)
        try:
            _adjoint(frames, p, True, ctx=ctx)
        except _lib.GtError as e:
            failed += 1
            assert e.status == _lib.GT_E_OOM, (after, str(e))
        finally:
            _inject(kind, 0)
        a = _adjoint(frames, p, True, ctx=ctx)
        for x, y in zip(want, [a.rows(), a.sigma(), a.origin(), a.jacobian()]):
            np.testing.assert_array_equal(x, y)
    assert failed >= (5 if kind else 10)
