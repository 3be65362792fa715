"""Runs of deskewed columns at their edges: outputs narrower than a run, one
column past whole runs, a plane or a column only, shifts a rounding away from a
whole number (neighbouring outputs whose input columns are not neighbours),
runs that are partly or wholly outside the input."""
import numpy as np
import pytest

import deskew_oracle as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 1, 1), (5, 2, 3), (8, 7, 4), (12, 9, 6), (260, 33, 20), (1028, 10, 5)])
@pytest.mark.parametrize("angle,dz,xy", [(32.45, 0.3, 0.108), (60.0, 0.2, 0.1), (60.0, 0.6, 0.1), (89.0, 0.1, 0.1)])
@pytest.mark.parametrize("reverse", [False, True])
def test_runs_vs_oracle(shape, angle, dz, xy, reverse):
    from petakit5d_amd import deskewFrame3D
    print(f"[deskew runs] {shape} angle={angle} dz={dz} reverse={reverse}", flush=True)
    vol = (np.random.default_rng(6).random(shape) * 1000).astype(np.float32)
    for crop in (False, True):
        got = deskewFrame3D(vol, angle, dz, xy, reverse, Crop=crop)
        ref = D.deskew(vol, angle, dz, xy, reverse, crop)
        assert got.shape == ref.shape
        # a + f (b - a) in float32: within a few ulps of the largest operand
        np.testing.assert_allclose(got, ref, rtol=0, atol=4e-7 * 1000 * 4)
