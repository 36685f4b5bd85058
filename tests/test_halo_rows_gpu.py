"""The halo loaders of the FP32 2-D, fused separable, ragged and 3-D tile kernels, for
rows of any length: narrower than one four-column group, one group more or
less than a tile of 128 or 64 columns, tiles that cross a row's end, against
the oracle at 1e-5 relative L2. Infinities next to the border check that
columns outside the image read as zeros, not as the neighbouring row."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SPATIAL = 1
WIDTHS = [1, 2, 3, 5, 63, 65, 126, 127, 129, 131, 257]


@pytest.mark.parametrize("w", WIDTHS)
@pytest.mark.parametrize("h", [2, 65])
@pytest.mark.parametrize("mode", [0, 1], ids=["default", "expand"])
def test_conv2_and_separable(af, rng, w, h, mode):
    x = rng.random((w, h, 2), dtype=np.float32)
    for f in (3, 5, 7, 9):
        t = rng.uniform(-1, 1, (f, f)).astype(np.float32)
        got = af.convolve2(x, t, mode, SPATIAL).to_numpy()
        assert oracle.rel_l2(got, oracle.convolve(x, t, 2, mode == 1)) <= 1e-5
    for cf, rf in ((3, 3), (17, 17), (5, 12)):
        c, r = rng.uniform(-1, 1, cf).astype(np.float32), rng.uniform(-1, 1, rf).astype(np.float32)
        got = af.convolve_sep(c, r, x, mode).to_numpy()
        assert oracle.rel_l2(got, oracle.convolve2_sep(c, r, x, mode == 1)) <= 1e-5


def test_ragged(af, rng):
    dims = [(w, 40 + 7 * k) for k, w in enumerate(WIDTHS)]
    sig = [rng.random(d, dtype=np.float32) for d in dims]
    flt = [rng.uniform(-1, 1, (3 + 2 * (k % 7), 3 + 2 * (k % 5))).astype(np.float32) for k in range(len(dims))]
    modes = [k % 2 for k in range(len(dims))]
    outs = af.convolve2_ragged(sig, flt, modes)
    for s, f, m, o in zip(sig, flt, modes, outs):
        assert oracle.rel_l2(o.to_numpy(), oracle.convolve(s, f, 2, m == 1)) <= 1e-5


def test_infinite_columns_stay_in_their_rows(af, rng):
    x = rng.random((131, 20), dtype=np.float32)
    x[0, 7] = x[130, 11] = np.inf
    t = rng.uniform(0.1, 1, (5, 5)).astype(np.float32)
    got = af.convolve2(x, t, 0, SPATIAL).to_numpy()
    ref = oracle.convolve(x, t, 2, False)
    np.testing.assert_array_equal(np.isinf(got), np.isinf(ref))
    assert not np.isnan(got).any()


@pytest.mark.parametrize("w", [1, 2, 3, 31, 33, 64, 67, 131])
@pytest.mark.parametrize("h,d", [(1, 2), (7, 9), (17, 8)])
@pytest.mark.parametrize("f", [3, 5])
def test_conv3(af, rng, w, h, d, f):
    x = rng.uniform(-1, 1, (w, h, d)).astype(np.float32)
    t = rng.uniform(0.1, 1, (f, f, f)).astype(np.float32)
    for mode in (0, 1):
        got = af.convolve3(x, t, mode, SPATIAL).to_numpy()
        assert oracle.rel_l2(got, oracle.convolve(x, t, 3, mode == 1)) <= 1e-5
    # infinities next to the volume's faces: columns, rows and planes outside
    # read as zeros, and no tap meets a value that is not its own
    x[0, 0, d - 1] = x[w - 1, h - 1, 0] = np.inf
    got, ref = af.convolve3(x, t, 0, SPATIAL).to_numpy(), oracle.convolve(x, t, 3, False)
    np.testing.assert_array_equal(np.isinf(got), np.isinf(ref))
    assert not np.isnan(got).any()


def test_conv2_rows_past_the_loader(af, rng):
    """Rows of 2^22 columns and more take the older loader, a last tile across
    the row's end included."""
    x = rng.random(((1 << 22) + 1, 3), dtype=np.float32)
    t = rng.uniform(-1, 1, (5, 5)).astype(np.float32)
    got = af.convolve2(x, t, 0, SPATIAL).to_numpy()
    assert oracle.rel_l2(got, oracle.convolve(x, t, 2, False)) <= 1e-5
    cut = slice((1 << 22) - 200, None)
    assert oracle.rel_l2(got[cut], oracle.convolve(x, t, 2, False)[cut]) <= 1e-5
