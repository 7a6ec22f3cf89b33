"""The streaming bandpass against the oracle where it can go wrong: every
smoothing radius, frames narrower than a strip and one column around its
edges (128 columns per wave, 256 per work item), frame bases at any multiple
of the element size, and uint16 boxcar sums past 2^24.

Bars as in test_gpu_parity: the same candidate pixels, positions within 1e-4
px, masses within 1e-5 relative.
"""
import numpy as np
import pytest

from tests.test_gpu_parity import _check, _oracle_movie
from tracking_optimizations_amd import _lib
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu

DTYPES = {"u8": np.uint8, "u16": np.uint16, "f32": np.float32}


def _noise(shape, dtype, seed):
    """Bright noise: uint16 near saturation, so that a window of k >= 17 rows
    sums past 2^24; float32 of both signs and uneven magnitudes."""
    rng = np.random.default_rng(seed)
    if dtype == "u8":
        return rng.integers(0, 256, shape, dtype=np.uint8)
    if dtype == "u16":
        return rng.integers(50000, 65536, shape, dtype=np.uint16)
    return (rng.standard_normal(shape) * np.exp(rng.uniform(-3, 6, shape))).astype(np.float32)


@pytest.mark.parametrize("dtype", sorted(DTYPES))
@pytest.mark.parametrize("k", [2, 3, 5, 8, 9, 11, 13, 15, 16, 17, 19, 21, 23, 25, 27, 29, 31, 33])
def test_radii_and_widths(dtype, k):
    import torch
    torch.cuda.init()   # before the first context of a process
    ctx = _lib.default_context(0)
    r = k // 2
    for n, (h, w) in enumerate([(max(r, 9), max(r, 2)), (29, 17), (37, 127), (31, 128), (33, 129),
                                (21, 255), (25, 257), (70, 131)]):
        frames = _noise((2, h, w), dtype, 100 * k + n)
        # a base one element past an allocation's start, odd frame sizes
        flat = torch.zeros(frames.size + 1, dtype=getattr(torch, {"u8": "uint8", "u16": "uint16",
                                                                 "f32": "float32"}[dtype]))
        flat[1:] = torch.from_numpy(frames.reshape(-1))
        dev = flat.cuda()[1:].reshape(2, h, w)
        for pct in (None, 30):
            kw = dict(diameter=5, separation=5, smoothing_size=k, percentile=pct)
            print(f"[bandpass] {dtype} k={k} {h}x{w} percentile={pct}", flush=True)
            rows, cand, _, _ = locate(dev, make_params(**kw), ctx=ctx)
            ref_rows, ref_cand = _oracle_movie(frames, kw)
            _check(rows, cand, ref_rows, ref_cand, f"{dtype}/k={k}/{h}x{w}/pct={pct}")


def test_long_segments_and_narrow_frames():
    """Rows per work item at both ends of the accepted range, and frames one
    and two pixels wide (the two-pass form and the narrowest streaming one)."""
    ctx = _lib.Context(0)
    frames = _noise((2, 300, 140), "u16", 7)
    kw = dict(diameter=5, separation=5, smoothing_size=9, percentile=40)
    ref = _oracle_movie(frames, kw)
    for seg in (16, 17, 272):
        ctx.set_launch_shape(seg)
        rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
        _check(rows, cand, *ref, f"seg={seg}")
    for w in (1, 2, 3):
        kw = dict(diameter=1, separation=2, smoothing_size=3)
        frames = _noise((2, 40, w), "u16", w)
        rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
        _check(rows, cand, *_oracle_movie(frames, kw), f"width {w}")
    ctx.close()


def _blocks_of_zeros(h, w, seed):
    # whole numbers: what is rounded stays above the denormals after scaling
    f = np.random.default_rng(seed).integers(-300, 700, (2, h, w)).astype(np.float32)
    f[:, 20:60, 30:90] = 0
    f[1, :, w - 40:] = 0
    return f


# float quotients come from a reciprocal where every lane's is in range, else
# from the division: zeros, values whose products with the reciprocal's low part
# are denormal (2^-100 and below), large ones.  A power of two scales every
# exact and every rounded step, so the rows are the same and the masses scale.
@pytest.mark.parametrize("exponent", [-110, -100, -92, -60, 60])
def test_float_range(exponent):
    ctx = _lib.default_context(0)
    frames = _blocks_of_zeros(131, 281, 5)
    kw = dict(diameter=5, separation=6, smoothing_size=5)
    ref = locate(frames, make_params(**kw), ctx=ctx)
    _check(ref[0], ref[1], *_oracle_movie(frames, kw), "zeros")
    scale = np.float32(2.0 ** exponent)
    got = locate(frames * scale, make_params(**kw), ctx=ctx)
    assert np.array_equal(got[1], ref[1])
    mass = [c[0] for c in ref[2]].index("mass")
    keep = [i for i in range(ref[0].shape[1]) if i != mass]
    assert np.array_equal(got[0][:, keep], ref[0][:, keep])
    assert np.array_equal(got[0][:, mass], ref[0][:, mass] * scale)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_float_not_finite(value):
    """One pixel that is not finite: rows out of its reach are untouched."""
    ctx = _lib.default_context(0)
    frames = _blocks_of_zeros(131, 281, 6)
    p = make_params(diameter=5, separation=6, smoothing_size=5)
    ref = locate(frames, p, ctx=ctx)
    frames[0, 90, 150] = value
    got = locate(frames, p, ctx=ctx)

    def far(r):
        away = (r[0][:, 0] != 0) | (np.abs(r[0][:, 2] - 90) > 40) | (np.abs(r[0][:, 3] - 150) > 40)
        return r[0][away], r[1][away]

    assert all(np.array_equal(a, b) for a, b in zip(far(got), far(ref)))


@pytest.mark.parametrize("dtype", ["u16", "f32"])
@pytest.mark.parametrize("noise_size", [0.3, 1.0, 2.0, 7.5])
def test_divisors(dtype, noise_size):
    """Widths of the Gaussian, each a divisor of its own; with 11 taps 2.0 is
    one whose rounded reciprocal misses a significand, so that a neighbour of
    its low part serves."""
    ctx = _lib.default_context(0)
    frames = _noise((2, 90, 140), dtype, 9)
    kw = dict(diameter=5, separation=5, smoothing_size=11, noise_size=noise_size)
    rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
    _check(rows, cand, *_oracle_movie(frames, kw), f"{dtype}/noise={noise_size}")
