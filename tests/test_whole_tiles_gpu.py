"""The 2-D tile kernel for 8- to 32-bit whole numbers against the oracle,
exactly: sizes around the 128 x 32 tile and narrower than one load, every
filter side it serves, both borders, every batch kind; and sums past the range
of the type, which must convert as in the general kernel (reached here with
the same filter in a larger, even-sided one)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SPATIAL = 1
TYPES = [np.uint8, np.int8, np.bool_, np.uint16, np.int16, np.int32, np.uint32]
SIZES = [(1, 2), (3, 40), (5, 31), (127, 33), (128, 32), (129, 65), (300, 7)]


def _raw(a):
    return a.view(np.int8) if a.dtype == np.bool_ else a


def _data(rng, shape, dt):
    if dt == np.bool_:
        return rng.integers(0, 2, shape).astype(dt)
    return rng.integers(0 if np.dtype(dt).kind == "u" else -50, 100, shape).astype(dt)


def _taps(rng, shape, dt):
    # positive for unsigned results, small enough that sums fit the type
    w = rng.random(shape) if np.dtype(dt).kind in "ub" else rng.uniform(-1, 1, shape)
    return (w / (shape[0] * shape[1] / 2.0)).astype(np.float32)


@pytest.mark.parametrize("f", [3, 5, 7, 9])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("mode", [0, 1], ids=["default", "expand"])
def test_sizes(af, rng, f, size, mode):
    for dt in (np.uint8, np.int16):
        x, w = _data(rng, size, dt), _taps(rng, (f, f), dt)
        got = af.convolve2(x, w, mode, SPATIAL).to_numpy()
        np.testing.assert_array_equal(got, oracle.convolve(x, w, 2, mode == 1))


@pytest.mark.parametrize("dt", TYPES, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("dims", [((150, 40, 3), (5, 5)), ((70, 35), (3, 3, 4)), ((33, 34, 2, 2), (7, 7, 2, 2))],
                         ids=["lhs", "rhs", "same"])
def test_types_and_batches(af, rng, dt, dims):
    x, w = _data(rng, dims[0], dt), _taps(rng, dims[1], dt)
    got = af.convolve2(x, w, 1, SPATIAL).to_numpy()
    np.testing.assert_array_equal(_raw(got), _raw(oracle.convolve(x, w, 2, True)))


@pytest.mark.parametrize("dt", TYPES, ids=lambda d: np.dtype(d).name)
def test_sums_past_the_range(af, rng, dt):
    x = _data(rng, (140, 37), dt)
    w = (rng.uniform(-1, 1, (5, 5)) * (1e9 if np.dtype(dt).itemsize == 4 else 3e3)).astype(np.float32)
    wide = np.zeros((6, 6), np.float32)
    wide[:5, :5] = w
    got = _raw(af.convolve2(x, w, 1, SPATIAL).to_numpy())
    ref = _raw(af.convolve2(x, wide, 1, SPATIAL).to_numpy())
    np.testing.assert_array_equal(got, ref[:-1, :-1])


def test_more_tiles_than_one_launch_takes(af, rng):
    # 2^24 and some images of one tile each: the general kernel's grid-stride loop
    few, times = 997, 16829
    base, w = rng.integers(0, 100, (few, 2, 2), dtype=np.uint8), _taps(rng, (3, 3), np.uint8)
    ref = oracle.convolve(np.asfortranarray(base.T), w, 2, False)
    img = np.tile(base.reshape(few, 4), (times, 1)).reshape(-1, 2, 2).T
    assert few * times > 1 << 24
    got = af.convolve2(img, w, 0, SPATIAL).to_numpy().T.reshape(times, -1)
    assert (got == ref.T.reshape(1, -1)).all()
