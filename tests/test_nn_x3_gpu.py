"""FP32 layers on the BF16 matrix cores in three parts per operand
(AFHIP_NN_X3=1) against FP64: sizes around the 64 x 64 tile and the 32-deep
slice, strides with phases (some without taps), dilation. The bar is half of
the 1e-6 that FP32 sums of these lengths stay below, plus: the error may not
exceed that of the FP32 kernels on the same data. Values that three parts do
not hold (infinities, NaNs, magnitudes from 2^32) must come out as from the
FP32 kernels, and tiles of nothing but tiny values to the bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

GEOMS = [
    ((8, 8, 32, 1), (1, 1, 32, 64), (1, 1), (0, 0), (1, 1)),
    ((13, 10, 33, 2), (3, 3, 33, 65), (1, 1), (1, 1), (1, 1)),
    ((20, 17, 3, 2), (5, 5, 3, 7), (1, 1), (2, 2), (1, 1)),
    ((28, 28, 40, 2), (3, 3, 40, 70), (2, 2), (1, 1), (1, 1)),
    ((25, 20, 16, 1), (3, 2, 16, 70), (6, 5), (0, 1), (1, 1)),
    ((27, 9, 100, 2), (3, 3, 100, 128), (1, 1), (2, 2), (2, 2)),
]


def _id(g):
    return "x{}_w{}_s{}_p{}_d{}".format(*["x".join(map(str, v)) for v in g])


def _both(af, X, W, DY, g):
    st, pd, dl = g[2:]
    y = af.convolve2NN(X, W, st, pd, dl)
    dx = af.convolve2GradientNN(DY, X, W, y, st, pd, dl, af.AF_CONV_GRADIENT_DATA)
    return y.to_numpy(), dx.to_numpy()


@pytest.mark.parametrize("g", GEOMS, ids=_id)
def test_against_fp64(af, rng, g, monkeypatch):
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    y64 = oracle.conv2_nn_direct_f64(x, w, *g[2:])
    dy = rng.standard_normal(y64.shape).astype(np.float32)
    dx64 = oracle.conv2_data_grad_direct_f64(dy, x, w, *g[2:])
    X, W, DY = af.Array(x), af.Array(w), af.Array(dy)
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    y, dx = _both(af, X, W, DY, g)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", "1")
    y1, dx1 = _both(af, X, W, DY, g)
    for got, one, ref in ((y, y1, y64), (dx, dx1, dx64)):
        e = oracle.rel_l2(got, ref)
        assert e <= 5e-7
        assert e <= oracle.rel_l2(one, ref) + 1e-8
        # pixels that no tap reaches are exact zeros
        assert np.array_equal(got[ref == 0], ref[ref == 0])


@pytest.mark.parametrize("what", ["x", "w", "all_tiny"])
def test_values_out_of_range(af, rng, what, monkeypatch):
    g = ((30, 26, 40, 2), (3, 3, 40, 70), (1, 1), (1, 1), (1, 1))
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    dy = rng.standard_normal((30, 26, 70, 2)).astype(np.float32)
    odd = [np.inf, -np.inf, np.nan, 3e38, -1e30, 1e-38, 1e-42, 2e-35]
    if what == "x":
        for k, v in enumerate(odd):
            x[3 * k, 25 - 3 * k, 5 * k, k % 2] = v
            dy[29 - 3 * k, 3 * k, 8 * k, k % 2] = v
    elif what == "w":
        w[1, 1, 3, 7], w[0, 2, 39, 69], w[2, 0, 0, 64] = np.inf, 1e-40, np.nan
    else:
        x *= np.float32(1e-33)
        dy *= np.float32(1e-33)
    X, W, DY = af.Array(x), af.Array(w), af.Array(dy)
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    got = _both(af, X, W, DY, g)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", "1")
    for a, b in zip(got, _both(af, X, W, DY, g)):
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        fin = np.isfinite(b)
        np.testing.assert_array_equal(a[~fin & ~np.isnan(b)], b[~fin & ~np.isnan(b)])
        if what != "x":  # every tile reads the odd value
            np.testing.assert_array_equal(a[fin], b[fin])
        else:
            np.testing.assert_allclose(a[fin], b[fin], rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("split", ["2", "4"])
@pytest.mark.parametrize("g", GEOMS, ids=_id)
def test_split_reduction(af, rng, g, split, monkeypatch):
    # partial tiles and their sum: phase padding, splits without slices in a
    # phase without taps, columns past the last whole tile
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    y64 = oracle.conv2_nn_direct_f64(x, w, *g[2:])
    dy = rng.standard_normal(y64.shape).astype(np.float32)
    dx64 = oracle.conv2_data_grad_direct_f64(dy, x, w, *g[2:])
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", split)
    for got, ref in zip(_both(af, af.Array(x), af.Array(w), af.Array(dy), g), (y64, dx64)):
        assert oracle.rel_l2(got, ref) <= 5e-7
        assert np.array_equal(got[ref == 0], ref[ref == 0])


@pytest.mark.parametrize("split", ["2", "4"])
def test_values_out_of_range_in_a_split(af, rng, split, monkeypatch):
    # only the splits that read an infinity or a NaN run in FP32
    g = ((30, 26, 70, 2), (3, 3, 70, 70), (1, 1), (1, 1), (1, 1))
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    dy = rng.standard_normal((30, 26, 70, 2)).astype(np.float32)
    for k, v in enumerate([np.inf, np.nan, -3e38, 1e12, -np.inf]):
        x[3 * k, 25 - 3 * k, 5 * k, k % 2] = v
        dy[29 - 3 * k, 3 * k, 8 * k, k % 2] = v
    w[1, 1, 3, 7] = 1e11
    X, W, DY = af.Array(x), af.Array(w), af.Array(dy)
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", split)
    got = _both(af, X, W, DY, g)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    for a, b in zip(got, _both(af, X, W, DY, g)):
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
        fin = np.isfinite(b)
        np.testing.assert_array_equal(a[~fin & ~np.isnan(b)], b[~fin & ~np.isnan(b)])
        np.testing.assert_allclose(a[fin], b[fin], rtol=2e-5, atol=2e-5)


def test_tiny_values_among_others(af, rng, monkeypatch):
    # values far below the others (a saturated softmax's gradient) leave the
    # tile on the three parts: they add nothing to its sums but the side to
    # which a tie is rounded, so next to no bit differs from zeros in their
    # place (from the FP32 kernels' sums half of the values do)
    g = ((30, 26, 40, 2), (3, 3, 40, 70), (1, 1), (1, 1), (1, 1))
    x = rng.standard_normal(g[0]).astype(np.float32)
    w = (rng.standard_normal(g[1]) * 0.1).astype(np.float32)
    dy = rng.standard_normal((30, 26, 70, 2)).astype(np.float32)
    at = [rng.random(a.shape) < 0.3 for a in (x, w, dy)]
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    out = []
    for tiny in (0.0, 1e-35, -3e-42):
        for a, i in zip((x, w, dy), at):
            a[i] = tiny
        out.append(_both(af, af.Array(x), af.Array(w), af.Array(dy), g))
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            assert (a != b).mean() < 1e-3
            np.testing.assert_allclose(a, b, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("scale", [1e-15, 1e-18, 3e-20, 1e-21])
def test_products_near_the_denormals(af, rng, scale, monkeypatch):
    # sums from 1e-30 down to a few denormal steps: rounded once, to FP32's
    # last place or to its smallest step
    g = ((30, 26, 40, 2), (3, 3, 40, 70), (1, 1), (1, 1), (1, 1))
    x = (rng.standard_normal(g[0]) * scale).astype(np.float32)
    w = (rng.standard_normal(g[1]) * scale).astype(np.float32)
    y64 = oracle.conv2_nn_direct_f64(x, w, *g[2:])
    dy = (rng.standard_normal(y64.shape) * scale).astype(np.float32)
    dx64 = oracle.conv2_data_grad_direct_f64(dy, x, w, *g[2:])
    size = oracle.conv2_nn_direct_f64(abs(x), abs(w), *g[2:]), oracle.conv2_data_grad_direct_f64(abs(dy), x, abs(w), *g[2:])
    monkeypatch.setenv("AFHIP_NN_X3", "1")
    for got, ref, s in zip(_both(af, af.Array(x), af.Array(w), af.Array(dy), g), (y64, dx64), size):
        assert (abs(got - ref) <= 2.0 ** -149 + 5e-7 * s).all()


@pytest.mark.parametrize("dims", [(9, 0), (0, 9), (0, 0)], ids=lambda d: "x".join(map(str, d)))
def test_no_pixels(af, rng, dims, monkeypatch):
    # padding alone makes outputs: all zeros, whichever kernel is asked for
    X = af.constant(0, dims + (40, 2))
    W = af.Array((rng.standard_normal((3, 3, 40, 70)) * 0.1).astype(np.float32))
    for x3 in ("1", None):
        monkeypatch.setenv("AFHIP_NN_X3", x3) if x3 else monkeypatch.delenv("AFHIP_NN_X3")
        y = af.convolve2NN(X, W, (1, 1), (2, 2), (1, 1))
        assert y.dims == tuple(d + 2 for d in dims) + (70, 2)
        assert not y.to_numpy().any()


@pytest.mark.parametrize("f", [3, 7], ids=["patch", "gemm"])
@pytest.mark.parametrize("env", [None, "AFHIP_NN_X3", "AFHIP_NN_WG"])
def test_results_of_another_type_are_refused(af, f, env, monkeypatch):
    # f32 arrays have f32 results; the three-part kernels store nothing else
    if env:
        monkeypatch.setenv(env, "1")
    X, W = af.constant(1, (20, 20, 32, 2)), af.constant(1, (f, f, 32, 64))
    Y = af.constant(1, (20, 20, 64, 2))
    geo = ((1, 1), (f // 2, f // 2), (1, 1))
    for t in (af.f16, af.bf16):
        for call in (lambda: af.convolve2NN(X, W, *geo, out_type=t),
                     lambda: af.convolve2NN(af.constant(1, (0, 20, 32, 2)), W, (1, 1), (f, f), out_type=t),
                     lambda: af.convolve2GradientNN(Y, X, W, Y, *geo, af.AF_CONV_GRADIENT_DATA, out_type=t),
                     lambda: af.convolve2GradientNN(Y, X, W, Y, *geo, af.AF_CONV_GRADIENT_FILTER, out_type=t)):
            with pytest.raises(af.AfError) as e:
                call()
            assert e.value.code == af.AF_ERR_TYPE
