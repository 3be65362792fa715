"""The row kernel of deskewRotateFrame3D at its edges: eight, four and one value
a lane give the same bits (a window that starts off a multiple of eight or four
rows takes the narrower), for one and two chunks of dim 1, runs of y that are
cut short and windows of a few columns; against the oracle as well."""
import numpy as np
import pytest

import deskew_oracle as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 40, 12), (260, 33, 9), (264, 33, 9), (67, 25, 14)])
@pytest.mark.parametrize("dz,reverse", [(0.2, False), (0.3, True), (0.5, False), (0.5, True)])
@pytest.mark.parametrize("u16", [False, True])
def test_windows_equal_the_whole(shape, dz, reverse, u16):
    import petakit5d_amd as pk
    print(f"[dsr rows] {shape} dz={dz} reverse={reverse} u16={u16}", flush=True)
    g = np.random.default_rng(5)
    v = np.asfortranarray((g.random(shape) * 5000).astype(np.uint16 if u16 else np.float32))
    kw = dict(reverse=reverse, save16bit=u16)
    full = np.asarray(pk.deskewRotateFrame3D(v, 32.45, dz, 0.108, **kw))
    ref = D.deskew_rotate(v.astype(np.float32), 32.45, dz, 0.108, reverse=reverse)
    assert full.shape == ref.shape
    # single: three blends of values below 5000 in FP32 (1e-5 of the range); uint16: one count at a rounding edge
    assert np.abs(full.astype(np.float64) - ref).max() <= (0.5 if u16 else 0) + 5000 * 1e-5
    n1, n2, n3 = full.shape
    for lo in [(1, 1, 1), (2, 4, 3), (5, 9, 1), (4, n2 - 2, n3 - 1)]:
        for hi in [(n1, n2, n3), (n1 - 1, min(n2, lo[1] + 7), n3), (min(n1, lo[0] + 7), min(n2, lo[1] + 8), lo[2])]:
            if all(h >= l for h, l in zip(hi, lo)):
                got = pk.deskewRotateFrame3D(v, 32.45, dz, 0.108, bbox=[*lo, *hi], **kw)
                want = full[lo[0] - 1:hi[0], lo[1] - 1:hi[1], lo[2] - 1:hi[2]]
                np.testing.assert_array_equal(got, want, err_msg=f"window {lo} {hi}")
