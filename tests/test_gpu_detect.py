"""Candidate slots and percentile lists of tiles that hold many: coarse levels
and plateaus, so that windows tie and whole rows of a tile are candidates, and
ranges of the percentile that hold a large part of the frame; partial tiles at
both edges.  The oracle's candidates, whole numbers, are the same; bars on the
rows as in test_gpu_parity."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check, _oracle_movie
from tracking_optimizations_amd import _lib
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu


def _coarse(h, w, seed):
    rng = np.random.default_rng(seed)
    blocks = rng.integers(0, 3, (2, (h + 5) // 6, (w + 8) // 9)) * 700
    f = np.repeat(np.repeat(blocks, 6, 1), 9, 2)[:, :h, :w]
    f[1] = (np.arange(w)[None, :] % 16 == 5) * 900 + (np.arange(h)[:, None] % 12 == 3) * 900
    return f.astype(np.uint16)


# one window of each kernel: by lanes (4 .. 16), by rows (18 .. 26), any size
@pytest.mark.parametrize("diameter,separation", [(3, 3), (5, 4), (7, 6), (9, 9), (11, 11), (7, 13),
                                                 (11, 18), (9, 20), (11, 30)])
@pytest.mark.parametrize("percentile", [None, 10, 60, 99])
def test_many_candidates(diameter, separation, percentile):
    ctx = _lib.default_context(0)
    for h, w in ((64, 48), (131, 149), (193, 97)):
        frames = _coarse(h, w, 10 * diameter + separation)
        kw = dict(diameter=diameter, separation=separation, percentile=percentile)
        ref = _oracle_movie(frames, kw)
        print(f"[detect] d={diameter} sep={separation} pct={percentile} {h}x{w}", flush=True)
        rows, cand, _, _ = locate(frames, make_params(**kw), ctx=ctx)
        _check(rows, cand, *ref, f"d={diameter}/sep={separation}/{percentile}/{h}x{w}")


@pytest.mark.parametrize("diameter,separation", [(3, 3), (9, 9), (7, 20), (11, 45)])
def test_dedup_blocks(diameter, separation):
    """81 frames of 9 x 9 tiles, more than have a wave each, are deduplicated
    in blocks of 2x2 tiles; a frame at a time (the per-frame path) tile by
    tile.  The rows are equal, and the first frame's are the oracle's."""
    ctx = _lib.default_context(0)
    rng = np.random.default_rng(separation)
    frames = rng.integers(0, 400, (81, 520, 400)).astype(np.uint16)
    frames[:, ::5, ::7] += 3      # ties in mass
    kw = dict(diameter=diameter, separation=separation, percentile=30)
    p = make_params(**kw)
    got = locate(frames, p, ctx=ctx)
    want = locate(frames, p, plain=True, ctx=ctx)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    first = want[0][:, 0] == 0
    _check(want[0][first], want[1][first], *_oracle_movie(frames[:1], kw), "one frame")


@pytest.mark.parametrize("separation", [2, 4, 9, 14, 25])
@pytest.mark.parametrize("spots", [(), ((30, 70), (110, 30)), ((20, 34),)])
@pytest.mark.parametrize("transpose", [False, True])
def test_masses_beyond_binary32(separation, spots, transpose):
    """Finite float32 pixels near the limit give disks of infinite mass and so a
    NaN in y (or x): near no other record, such a row is kept wherever it
    lies, alone in its tile or block or beside finite ones."""
    f = np.zeros((1, 150, 170), np.float32)
    for y, x in ((20, 20), (40, 60), (100, 100)):
        for i, j in ((4, 0), (3, -2), (3, 2), (0, 0), (0, 4)):
            f[0, y + i, x + j] = 8e37
        f[0, y, x] *= 1.02
    for y, x in spots:
        f[0, y, x] = 50
    if transpose:
        f = np.ascontiguousarray(f.transpose(0, 2, 1))
    kw = dict(diameter=9, separation=separation, smoothing_size=3, noise_size=0.05)
    ref, ref_cand = _oracle_movie(f, kw)
    assert np.isnan(ref[:, 2:4]).any(axis=1).sum() >= 3 and np.isinf(ref[:, 1]).any()
    ctx = _lib.default_context(0)
    for fused in (True, False):
        ctx.set_fused_walk(fused)
        try:
            rows, cand, _, _ = locate(f, make_params(**kw), ctx=ctx)
        finally:
            ctx.set_fused_walk(True)
        np.testing.assert_array_equal(cand, ref_cand)
        np.testing.assert_allclose(rows, ref, rtol=1e-5, atol=1e-4)
