"""The two-dimensional register-FFT route of af_fft_convolve2 (real data,
padded sides 64..4096) against the oracle's restatement: each transform
length (every mix of radices 8, 4 and 2), both directions of the pair packing
(odd and even row counts), every batch kind, and lengths just below and at
the route's limits.

Bars as in test_fftconv_gpu.py: FP32 within 1e-5 relative L2, FP64 within
1e-12, integer results of integer data exact."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

DEFAULT, EXPAND = 0, 1

# (signal dims, filter dims): padded sides 64..4096 along dim0 and dim1
CASES = [
    ((41, 63), (9, 2)),               # 64 x 64, L1 exactly full
    ((60, 100), (5, 29)),             # 64 x 128 full: 60+5-1, 100+29-1
    ((97, 250), (33, 8)),             # 256 x 512, even filter side
    ((500, 90), (14, 40)),            # 1024 x 256
    ((1001, 33), (1100, 32)),         # 4096 x 64, filter longer than the signal
    ((1500, 77), (31, 31)),           # 2048 x 128
    ((50, 3000), (20, 31)),           # 128 x 4096
    ((65, 63, 5), (8, 7)),            # LHS, one filter spectrum for all
    ((70, 71), (9, 6, 3)),            # RHS
    ((70, 64, 2, 3), (9, 30, 2, 3)),  # SAME
]


def _id(c):
    return f"s{'x'.join(map(str, c[0]))}_f{'x'.join(map(str, c[1]))}"


def _run(af, x, w, mode):
    X, W = af.Array(x), af.Array(w)
    return af._out(af.lib().af_fft_convolve2, X.handle, W.handle, mode).to_numpy()


@pytest.mark.parametrize("case", CASES, ids=_id)
@pytest.mark.parametrize("mode", [DEFAULT, EXPAND], ids=["default", "expand"])
@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int32], ids=lambda d: np.dtype(d).name)
def test_lengths_and_kinds(af, rng, case, mode, dt):
    sd, fd = case
    if dt == np.int32:
        x, w = rng.integers(-9, 10, sd).astype(dt), rng.integers(-3, 4, fd).astype(dt)
    else:
        x, w = rng.standard_normal(sd).astype(dt), rng.standard_normal(fd).astype(dt)
    got = _run(af, x, w, mode)
    ref = oracle.fft_convolve(x, w, 2, mode == EXPAND)
    assert got.shape == ref.shape and got.dtype == ref.dtype
    if dt == np.int32:
        np.testing.assert_array_equal(got, ref)
    else:
        assert oracle.rel_l2(got, ref) <= (1e-12 if dt == np.float64 else 1e-5)


@pytest.mark.parametrize("dt", [np.uint8, np.int8, np.int16, np.uint16, np.uint32, np.int64, np.uint64],
                         ids=lambda d: np.dtype(d).name)
def test_integer_storage(af, rng, dt):
    x, w = rng.integers(0, 3, (101, 67)).astype(dt), rng.integers(0, 2, (7, 6)).astype(dt)
    got = _run(af, x, w, EXPAND)
    ref = oracle.fft_convolve(x, w, 2, True)
    np.testing.assert_array_equal(got, ref)


def test_nan_stays_in_its_slice(af, rng):
    x = rng.standard_normal((80, 75, 3)).astype(np.float32)
    w = rng.standard_normal((20, 21)).astype(np.float32)
    clean = _run(af, x, w, DEFAULT)
    x[11, 12, 1] = np.nan
    got = _run(af, x, w, DEFAULT)
    assert np.isnan(got[:, :, 1]).all()
    np.testing.assert_array_equal(got[:, :, [0, 2]], clean[:, :, [0, 2]])
