"""Rotations that keep dim-1 rows: the four-column kernel (four rows and one
row a lane) gives the bits of the general one, infinities and NaN included, and
the extents of the projection found on the device are numpy's."""
import ctypes
import math

import numpy as np
import pytest

from petakit5d_amd.rotate import rotate_transform

pytestmark = pytest.mark.gpu


def _warp(t, inv, od):
    import torch
    from petakit5d_amd import _lib
    ctx = _lib.default_context()
    out = torch.full((od[2], od[1], od[0]), 7.0, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    inv = np.ascontiguousarray(inv)
    ctx.check(_lib.load().pk_affine_warp3d(
        ctx.handle, ctypes.c_void_p(t.data_ptr()), _lib.i64x3(tuple(t.shape)[::-1]),
        inv.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), _lib.i64x3(od), ctypes.c_void_p(out.data_ptr())))
    return out.cpu().numpy()


@pytest.mark.parametrize("shape", [(64, 40, 12), (260, 33, 9), (67, 25, 14), (3, 9, 5), (1, 2, 1)])
@pytest.mark.parametrize("rows", [0, -1, 2])  # output rows beyond the input's
def test_equal_to_the_general_kernel(shape, rows):
    import torch
    ny, nx, nz = shape
    od = (max(ny + rows, 1), nx + 11, 2 * nz + 7)
    print(f"[rotate rows] {shape} -> {od}", flush=True)
    g = np.random.default_rng(7)
    v = (g.standard_normal((nz, nx, ny)) * 100).astype(np.float32)
    if ny > 3:
        v[g.random(v.shape) < 1e-3] = np.nan
        v[g.random(v.shape) < 1e-3] = np.inf
    t = torch.from_numpy(v).cuda()
    ct, st, zx = math.cos(0.55), math.sin(0.55), 1.7
    m = np.array([[ct, 0, -st / zx, 0], [0, 1, 0, 0], [st, 0, ct / zx, 0], [-0.3 * nx, 0, 0.2 * nz, 1]])
    general = m.copy()
    general[0, 1] = 1e-300  # no row moves by it, but the entry is not 0
    np.testing.assert_array_equal(_warp(t, m, od), _warp(t, general, od))


@pytest.mark.parametrize("ny", [1, 64, 300])
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("kind", ["sheared", "negative", "constant", "zero"])
def test_extents(ny, reverse, kind):
    """Columns with a positive value only at the end, only negative values,
    negative values and a zero, NaN, and projections without an edge."""
    import torch
    import petakit5d_amd as pk
    print(f"[extents] ny={ny} reverse={reverse} {kind}", flush=True)
    nx, nz, zx = 90, 21, 2.3
    g = np.random.default_rng(ny)
    v = np.zeros((ny, nx, nz), np.float32)
    if kind == "constant":
        v[:] = 2.0
    for p in range(nz if kind in ("sheared", "negative") else 0):
        v[-1, 2 * p:2 * p + 40, p] = 1.0
        if kind == "negative":  # max: a negative number (true) where no value is 0, else 0 (false)
            v[:, 2 * p:2 * p + 40, p] = -g.random((ny, 40)) - 0.5
            v[0, 2 * p, p] = 0.0
            v[-1, 2 * p + 39, p] = np.nan
    want = rotate_transform(v.shape, 31.5, zx, reverse, proj=v.max(axis=0))
    t = torch.from_numpy(v.transpose(2, 1, 0).copy()).cuda().permute(2, 1, 0)
    out = pk.rotateFrame3D(t, 31.5, zx, reverse)
    assert tuple(out.shape) == want[1]
