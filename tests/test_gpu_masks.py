"""The edge masks' kernels at the edges of their ranges: the whole-volume mask
on bits (rows of one word, one short of and past a word, 64 words; the largest
ball of the bit form and the first of the searches) against scipy's exact
distance transform, and the mask of a chunk (full rectangle and not) against
the oracle.  Whole numbers: equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _holes(shape, seed, frac):
    g = np.random.default_rng(seed)
    return np.asfortranarray(np.where(g.random(shape) < frac, 0, g.integers(1, 60000, shape)).astype(np.uint16))


@pytest.mark.parametrize("shape", [(1, 6, 5), (63, 40, 9), (64, 7, 30), (65, 33, 3), (130, 61, 57), (200, 90, 70),
                                   (4096, 9, 7), (4097, 6, 5)])
@pytest.mark.parametrize("E", [1, 2, 8, 24, 25])
def test_whole_volume_mask(shape, E):
    from scipy import ndimage as ndi
    from petakit5d_amd.chunks import edge_erosion_mask
    print(f"[edge mask] {shape} E={E}", flush=True)
    im = _holes(shape, E, 2e-4)
    bw = np.zeros(shape, bool)
    bw[1:-1, 1:-1, 1:-1] = (im > 0)[1:-1, 1:-1, 1:-1]
    d = ndi.distance_transform_edt(bw)
    want = np.rint(d * d).astype(np.int64) > (E - 1) ** 2
    np.testing.assert_array_equal(edge_erosion_mask(im, E), want)
    f = im.astype(np.float32)
    f[im == 0] = np.where(np.arange(f[im == 0].size) % 2, -1.0, np.nan)  # not > 0 either way
    np.testing.assert_array_equal(edge_erosion_mask(f, E), want)


@pytest.mark.parametrize("shape", [(32, 30, 27), (45, 20, 18), (72, 24, 16)])
@pytest.mark.parametrize("E", [1, 3, 8])
@pytest.mark.parametrize("full", [True, False])
def test_chunk_mask(oracle, shape, E, full):
    """One iteration with EdgeErosion: zero exactly where the oracle's mask is."""
    import petakit5d_amd as pk
    print(f"[chunk mask] {shape} E={E} full={full}", flush=True)
    im = _holes(shape, 3, 0.0 if full else 0.01)
    im[im > 0] |= 1024  # the result stays positive inside the mask
    psf = np.zeros((3, 3, 3), np.float32)
    psf[1, 1, 1] = 1
    mask = oracle.decon_mask_edge_erosion(im != 0, E)
    got, _, _ = pk.decon_lucy_function(im.astype(np.float32), psf, 1, Background=0, save16bit=False, EdgeErosion=E)
    np.testing.assert_array_equal(np.asarray(got) > 0, mask & (im > 0))
