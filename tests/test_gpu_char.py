"""Characterisation columns against the oracle over disk sizes: radii 0 to 15,
even diameters (host and shader disks differ), fewer taps than accumulators
and every remainder of eight, row counts that leave the last group of eight
lanes and the last workgroup partly idle, next to the raw signal columns.

Bars as in test_gpu_parity (1e-5 relative, the same non-finite entries)."""
import numpy as np
import pytest

from tests.test_gpu_parity import _check, _oracle_movie
from tracking_optimizations_amd import _lib
from tracking_optimizations_amd.gpu_tracking import locate, make_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["u8", "u16", "f32"])
@pytest.mark.parametrize("diameter", [1, 2, 3, 4, 5, 6, 8, 9, 11, 14, 16, 17, 21, 24, 31])
def test_columns_over_diameters(dtype, diameter):
    ctx = _lib.default_context(0)
    rng = np.random.default_rng(diameter)
    frames = rng.integers(0, 200, (3, 131, 157))
    frames = {"u8": frames.astype(np.uint8), "u16": (frames * 300).astype(np.uint16),
              "f32": (frames * 0.63).astype(np.float32)}[dtype]
    for cpu, gpu in ((True, False), (False, True), (True, True)):
        kw = dict(diameter=diameter, separation=max(diameter, 3), smoothing_size=max(diameter, 3) | 1,
                  characterize=gpu, cpu_processed=cpu)
        print(f"[char] {dtype} d={diameter} cpu={cpu} gpu={gpu}", flush=True)
        rows, cand, cols, _ = locate(frames, make_params(**kw), ctx=ctx)
        ref = _oracle_movie(frames, kw)
        assert len(ref[1]) > 10
        _check(rows, cand, *ref, f"{dtype}/d={diameter}/cpu={cpu}/gpu={gpu}")
    # the raw signal columns lie between the two groups
    raw, _, rcols, _ = locate(frames, make_params(**kw, sig_radius=2.0, bg_radius=5.0), ctx=ctx)
    names, rnames = [n for n, _ in cols], [n for n, _ in rcols]
    for n in names:
        np.testing.assert_array_equal(raw[:, rnames.index(n)], rows[:, names.index(n)], err_msg=n)
