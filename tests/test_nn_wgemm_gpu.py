"""The filter gradient from channel-last copies (AFHIP_NN_WG=1) against FP64:
filters and channels around the 64 x 64 tile and the 32-channel slice, tap
counts that do and do not fill groups of three, fewer pixels than a slice,
rows shorter than a slice and images that end inside one, strides, padding
beyond the filter and dilation.

Bars: 16-bit operands with FP32 results as FP32 sums of exact products, 2e-6
relative L2 of FP64 on the rounded operands; FP32 5e-7, and no worse than the
element gather on the same data; results for values outside the range of the
three-part form as from the element gather."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# (x dims [W,H,C,N], w dims [fw,fh,C,K], stride, pad, dilation)
GEOMS = [
    ((3, 3, 5, 1), (3, 3, 5, 4), (1, 1), (0, 0), (1, 1)),          # one output pixel
    ((8, 8, 64, 1), (1, 1, 64, 64), (1, 1), (0, 0), (1, 1)),
    ((13, 10, 33, 2), (3, 3, 33, 65), (1, 1), (1, 1), (1, 1)),
    ((5, 4, 70, 7), (2, 2, 70, 31), (1, 1), (1, 0), (1, 1)),       # images of 15 pixels
    ((27, 21, 40, 2), (5, 5, 40, 36), (2, 3), (2, 1), (1, 1)),
    ((40, 30, 3, 3), (3, 1, 3, 130), (1, 1), (3, 0), (1, 1)),      # padding beyond the filter
    ((33, 18, 96, 2), (3, 3, 96, 32), (1, 2), (2, 2), (2, 3)),
]


def _id(g):
    return "x{}_w{}_s{}_p{}_d{}".format(*["x".join(map(str, v)) for v in g])


def _data(rng, g):
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    yd = tuple(1 + (g[0][i] + 2 * g[3][i] - ((g[1][i] - 1) * g[4][i] + 1)) // g[2][i] for i in (0, 1))
    dy = rng.standard_normal(yd + (g[1][3], g[0][3])).astype(np.float32)
    return x, w, dy


def _dw(af, X, W, DY, g, t):
    y = af.constant(0, DY.dims, t)
    return af.convolve2GradientNN(DY, X, W, y, *g[2:], af.AF_CONV_GRADIENT_FILTER, out_type=af.f32).to_numpy()


@pytest.mark.parametrize("dt,bar", [("f32", 5e-7), ("bf16", 2e-6), ("f16", 2e-6)], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("g", GEOMS, ids=_id)
def test_against_fp64(af, rng, g, dt, bar, monkeypatch):
    t = {"bf16": af.bf16, "f16": af.f16, "f32": af.f32}[dt]
    X, W, DY = (af.Array(a).astype(t) for a in _data(rng, g))
    ref = oracle.conv2_filter_grad_direct_f64(*(a.astype(af.f32).to_numpy() for a in (DY, X, W)), *g[2:])
    monkeypatch.setenv("AFHIP_NN_WG", "1")
    e = oracle.rel_l2(_dw(af, X, W, DY, g, t), ref)
    assert e <= bar
    if dt == "f32":
        monkeypatch.setenv("AFHIP_NN_GATHER", "1")
        assert e <= oracle.rel_l2(_dw(af, X, W, DY, g, t), ref) + 1e-8


def test_16_bit_results(af, rng, monkeypatch):
    g = GEOMS[2]
    x, w, dy = _data(rng, g)
    monkeypatch.setenv("AFHIP_NN_WG", "1")
    for t, bar in ((af.bf16, 1e-2), (af.f16, 2e-3)):
        X, W, DY = (af.Array(a).astype(t) for a in (x, w, dy))
        got = af.convolve2GradientNN(DY, X, W, af.constant(0, DY.dims, t), *g[2:], af.AF_CONV_GRADIENT_FILTER)
        assert got.type == t
        assert oracle.rel_l2(got.astype(af.f32).to_numpy(), oracle.conv2_filter_grad_direct_f64(dy, x, w, *g[2:])) <= bar


@pytest.mark.parametrize("what", ["spots", "all_tiny"])
def test_values_out_of_range(af, rng, what, monkeypatch):
    g = ((30, 26, 40, 2), (3, 3, 40, 70), (1, 1), (1, 1), (1, 1))
    x, w, dy = _data(rng, g)
    if what == "spots":
        x[3, 4, 5, 0], x[20, 11, 17, 1], x[7, 7, 30, 1] = np.inf, 1e-42, 3e38
        dy[9, 9, 66, 1], dy[2, 20, 3, 0] = np.nan, -1e-38
    else:
        x *= np.float32(1e-33)
    X, W, DY = af.Array(x), af.Array(w), af.Array(dy)
    monkeypatch.setenv("AFHIP_NN_WG", "1")
    a = _dw(af, X, W, DY, g, af.f32)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    b = _dw(af, X, W, DY, g, af.f32)
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    fin = np.isfinite(b)
    np.testing.assert_array_equal(a[~fin & ~np.isnan(b)], b[~fin & ~np.isnan(b)])
    assert oracle.rel_l2(a[fin], b[fin]) <= 2e-6


@pytest.mark.parametrize("taps", [(1, 1), (2, 1), (1, 3), (2, 2), (5, 1), (4, 4)], ids=lambda t: "x".join(map(str, t)))
@pytest.mark.parametrize("dt,bar", [("f32", 5e-7), ("bf16", 2e-6)], ids=["f32", "bf16"])
def test_tap_groups(af, rng, taps, dt, bar, monkeypatch):
    # counts that run tap by tap and in threes, over more than one channel tile
    t = {"bf16": af.bf16, "f32": af.f32}[dt]
    g = ((19, 23, 70, 3), taps + (70, 66), (1, 2), (1, 0), (1, 1))
    X, W, DY = (af.Array(a).astype(t) for a in _data(rng, g))
    ref = oracle.conv2_filter_grad_direct_f64(*(a.astype(af.f32).to_numpy() for a in (DY, X, W)), *g[2:])
    monkeypatch.setenv("AFHIP_NN_WG", "1")
    assert oracle.rel_l2(_dw(af, X, W, DY, g, t), ref) <= bar
