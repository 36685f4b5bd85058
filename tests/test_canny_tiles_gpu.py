"""af_canny's tile kernels against the oracle's restatement, exactly: sizes
around the 64 x 16 tile (one tile, one past it, many, narrower than a tile),
edges that cross many tiles (a spiral, whose weak pixels hang on one seed),
thresholds that make every pixel weak (so that the linear-offset neighbours
wrap from one column to the next), batches, more tiles than one workgroup
reduces, and each storage type."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _check(af, img, ct, lo, hi, fast=False):
    g = af.canny(img, ct, lo, hi, 3, fast).to_numpy().astype(np.uint8)
    np.testing.assert_array_equal(g, oracle.canny(img, ct, lo, hi, 3, fast))


def _blobs(shape, seed):
    import scipy.ndimage as ndi

    rng = np.random.default_rng(seed)
    x = ndi.gaussian_filter(rng.random(shape), (1.5, 1.5) + (0,) * (len(shape) - 2)) * 255.0
    return x + (rng.random(shape) > 0.99) * 60.0


SIZES = [(5, 5), (6, 40), (64, 16), (65, 17), (63, 33), (130, 50), (200, 6), (40, 130, 2), (66, 18, 2, 2)]


@pytest.mark.parametrize("shape", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("lo,hi", [(0.1, 0.3), (0.02, 0.6), (0.0, 0.9), (0.5, 0.0)])
@pytest.mark.parametrize("fast", [False, True], ids=["l2", "l1"])
def test_sizes_and_thresholds(af, shape, lo, hi, fast):
    _check(af, _blobs(shape, 20261210).astype(np.float32), 0, lo, hi, fast)


@pytest.mark.parametrize("shape", [(65, 17), (150, 70), (40, 60, 3)], ids=lambda s: "x".join(map(str, s)))
def test_otsu(af, shape):
    _check(af, _blobs(shape, 20261211).astype(np.float32), 1, 0.4, 0.0)


def test_spiral_from_one_seed(af):
    # a step edge of low contrast along a spiral; one stretch of it rises to
    # a contrast that passes the high threshold
    n = 200
    img = np.zeros((n, n), np.float32)
    for k, lo in enumerate(range(6, 90, 8)):
        img[lo:n - lo, lo:n - lo] = 20.0 * (k % 2 == 0)
    for lo in range(6, 82, 8):  # joins one ring to the next
        img[lo:lo + 8, 100:104] = 20.0 * ((lo - 6) // 8 % 2 == 1)
    img[6:14, :] *= 1.0 + 2.0 * np.exp(-((np.arange(n) - 40.0) / 20.0) ** 2).astype(np.float32)
    ref = oracle.canny(img, 0, 0.1, 0.8)
    assert ref.sum() > 2000
    np.testing.assert_array_equal(af.canny(img, 0, 0.1, 0.8).to_numpy().astype(np.uint8), ref)


def test_more_tiles_than_one_workgroup_reduces(af):
    # 1100 slices of one tile; the largest value lies in the last
    rng = np.random.default_rng(20261212)
    img = (rng.random((12, 9, 40, 28)) * 100).astype(np.float32)
    img[5, 4, 39, 27] = 900.0
    _check(af, img, 0, 0.05, 0.15)


@pytest.mark.parametrize("dt", [np.float64, np.int32, np.uint32, np.int16, np.uint16, np.int8, np.uint8],
                         ids=lambda d: np.dtype(d).name)
def test_storage_types(af, dt):
    _check(af, (_blobs((70, 40), 20261213) * 0.4).astype(dt), 0, 0.1, 0.3)


def test_nan_and_inf(af):
    img = _blobs((80, 50), 20261214).astype(np.float32)
    img[20, 10] = np.inf
    img[60, 40] = np.nan
    _check(af, img, 0, 0.1, 0.3)


@pytest.mark.parametrize("otsu", [0, 1], ids=["manual", "otsu"])
def test_more_tiles_than_one_launch_takes(af, otsu):
    # 2^24 and some images of one tile each; a launch holds fewer workgroups
    few, times = 997, 16829
    rng = np.random.default_rng(20261215)
    base = rng.integers(0, 9, (few, 5, 5), dtype=np.uint8)
    ref = oracle.canny(np.asfortranarray(base.T), otsu, 0.2, 0.5)
    assert few * times > 1 << 24 and 0 < ref.mean() < 1
    img = np.tile(base.reshape(few, 25), (times, 1)).reshape(-1, 5, 5).T
    got = af.canny(img, otsu, 0.2, 0.5).to_numpy().view(np.uint8).T.reshape(times, -1)
    assert (got == np.asarray(ref, np.uint8).T.reshape(1, -1)).all()
