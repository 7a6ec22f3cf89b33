"""Dilation windows of 16 to 64 pixels and disk radii up to 16 against the
oracle: every window that no kernel of its own serves, both of its starting
spans, walks inside detect and in the refine kernel, with and without a
percentile; frames a few tiles large with partial tiles, and smaller than one
window.

Bars as in test_gpu_parity."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check, _oracle_movie
from tracking_optimizations_amd import _lib
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu


def _movie(h, w, sigma, seed):
    rng = np.random.default_rng(seed)
    yy, xx = np.mgrid[:h, :w]
    f = rng.poisson(80, (2, h, w)).astype(np.float64)
    for k in range(max(3, h * w // 1500)):
        y, x, a = rng.uniform(0, h), rng.uniform(0, w), rng.uniform(200, 1500)
        f[k % 2] += a * np.exp(-((yy - y) ** 2 + (xx - x) ** 2) / (2 * sigma ** 2))
    return np.minimum(f, 65535).astype(np.uint16)


# (diameter, separation): windows trunc(2 sep / sqrt 2) = 28 .. 63, and 16 ..
# 26 with disks wider than their own kernels walk; 64 goes through a plane
@pytest.mark.parametrize("diameter,separation", [
    (3, 20), (5, 21), (7, 22), (9, 23), (11, 24), (13, 25), (15, 26), (17, 27), (19, 28),
    (21, 22), (21, 29), (23, 24), (23, 30), (25, 26), (27, 28), (29, 30), (31, 32), (31, 33),
    (32, 34), (9, 36), (15, 39), (31, 41), (31, 44), (5, 45), (11, 46),
    (17, 12), (19, 13), (23, 15), (31, 16), (21, 18), (20, 19), (33, 34),
])
def test_windows_and_radii(diameter, separation):
    ctx = _lib.default_context(0)
    for h, w in ((150, 203), (67, 49)):
        frames = _movie(h, w, 0.2 * diameter + 0.5, 100 * diameter + separation)
        for pct in (None, 60):
            kw = dict(diameter=diameter, separation=separation, percentile=pct,
                      smoothing_size=min(diameter, 33) | 1)
            ref = _oracle_movie(frames, kw)
            for fused in (True, False):
                print(f"[wide] d={diameter} sep={separation} {h}x{w} pct={pct} fused={fused}", flush=True)
                ctx.set_fused_walk(fused)
                try:
                    rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
                finally:
                    ctx.set_fused_walk(True)
                _check(rows, cand, *ref, f"d={diameter}/sep={separation}/{h}x{w}/{pct}/{fused}")


def _spots_and_bad_pixels(value):
    """Float32 spots on zeros, and a pixel of `value` 14 pixels from each: in its
    window from separation 20 on, out of reach of its disk and of its filter."""
    yy, xx = np.mgrid[:150, :203]
    f = np.zeros((1, 150, 203), np.float32)
    bad = []
    for k, (y, x) in enumerate(((40, 40), (41, 95), (40, 150), (104, 70), (105, 131))):
        r2 = (yy - y) ** 2 + (xx - x) ** 2
        f[0] += np.where(r2 <= 16, (300 + 20 * k) * np.exp(-r2 / 6.0), 0).astype(np.float32)
        bad.append((0, y + (0, 14, 0, -14, 10)[k], x + (14, 0, -14, 0, 10)[k]))
    g = f.copy()
    for b in bad:
        g[b] = value
    return f, g


@pytest.mark.parametrize("separation", [20, 22, 23, 30, 44, 45, 46])   # windows 28 .. 63, 65
@pytest.mark.parametrize("value", [np.nan, -np.nan, np.inf, -np.inf])
def test_not_finite_pixels_hide_no_neighbour(separation, value):
    """Windows without a kernel of their own skip NaN: the rows are those of the
    frame without the pixels; a percentile that is NaN leaves none."""
    ctx = _lib.default_context(0)
    clean, frames = _spots_and_bad_pixels(np.float32(value))
    for pct in (None, 60):
        kw = dict(diameter=9, separation=separation, percentile=pct)
        ref = _oracle_movie(clean, kw)
        assert len(ref[0]) >= 3
        for fused in (True, False):
            ctx.set_fused_walk(fused)
            try:
                rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
                none, _, _, _ = locate(frames, make_params(**{**kw, "percentile": 99.5}), ctx=ctx)
            finally:
                ctx.set_fused_walk(True)
            _check(rows, cand, *ref, f"sep={separation}/{value}/{pct}/{fused}")
            assert len(none) == 0
