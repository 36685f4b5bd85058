"""The channel-last GEMM (afhip_k_conv2_nn_gemm_split) against the element
gather, bit for bit: both walk the same 32-deep slices in the same order, so
the sums are equal whatever the tile. Sizes at its edges: output channels
around 64 and 128 rows per tile, odd numbers of slices per tap and per split
(a 16-bit stage holds two), pixels around a tile of 128 columns, image planes
that are and are not multiples of four pixels (vector stores), dilation, and
strides with many phases, some without taps. And against FP64."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# (x dims [W,H,C,N], w dims [fw,fh,C,K], stride, pad, dilation, splits)
GEOMS = [
    ((16, 8, 32, 1), (1, 1, 32, 64), (1, 1), (0, 0), (1, 1), 1),     # one slice, one column tile
    ((13, 10, 96, 1), (3, 3, 96, 65), (1, 1), (1, 1), (1, 1), 2),    # three slices per tap
    ((9, 7, 33, 3), (5, 5, 33, 128), (1, 1), (2, 2), (1, 1), 3),
    ((12, 11, 160, 2), (3, 1, 160, 129), (1, 1), (1, 0), (1, 1), 4),
    ((27, 9, 20, 2), (3, 3, 20, 200), (1, 1), (2, 2), (2, 2), 5),
    ((23, 21, 40, 2), (5, 5, 40, 36), (5, 5), (2, 2), (1, 1), 1),    # 25 phases
    ((25, 20, 16, 1), (3, 2, 16, 70), (6, 5), (0, 1), (1, 1), 2),    # phases without taps
    ((30, 30, 24, 2), (4, 4, 24, 24), (4, 4), (0, 0), (3, 3), 1),
]


def _id(g):
    return "x{}_w{}_s{}_p{}_d{}_n{}".format(*["x".join(map(str, v)) for v in g[:5]], g[5])


@pytest.mark.parametrize("dt,bar", [("f32", 1e-5), ("bf16", 1e-2), ("f16", 2e-3)], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("g", GEOMS, ids=_id)
def test_same_bits_as_element_gather(af, rng, g, dt, bar, monkeypatch):
    xd, wd, st, pd, dl, ns = g
    t = {"bf16": af.bf16, "f16": af.f16, "f32": af.f32}[dt]
    x = rng.standard_normal(xd).astype(np.float32)
    w = (rng.standard_normal(wd) * np.sqrt(2.0 / (wd[0] * wd[1] * wd[2]))).astype(np.float32)
    X, W = af.Array(x).astype(t), af.Array(w).astype(t)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", str(ns))

    def both():
        y = af.convolve2NN(X, W, st, pd, dl, out_type=af.f32)
        dy = np.random.default_rng(7).standard_normal(y.dims).astype(np.float32)
        DY = af.Array(dy).astype(t)
        dx = af.convolve2GradientNN(DY, X, W, y, st, pd, dl, af.AF_CONV_GRADIENT_DATA, out_type=af.f32)
        return y.to_numpy(), dx.to_numpy(), dy

    y, dx, dy = both()
    monkeypatch.setenv("AFHIP_NN_CL", "0")
    y1, dx1, _ = both()
    np.testing.assert_array_equal(y, y1)
    np.testing.assert_array_equal(dx, dx1)
    assert oracle.rel_l2(y, oracle.conv2_nn_direct_f64(x, w, st, pd, dl)) <= bar
    assert oracle.rel_l2(dx, oracle.conv2_data_grad_direct_f64(dy, x, w, st, pd, dl)) <= bar


# Results of an unsplit launch leave through LDS. Planes of whole and of broken
# groups of four pixels, channels one more than and less than a tile's rows,
# and enough columns for the 64 x 128 and 128 x 128 tiles (FP32 results of the
# latter leave in two halves).
STORES = [
    ((20, 12, 32, 2), (3, 3, 32, 65), (1, 1), (1, 1), (1, 1)),     # 64 x 64, 240-pixel planes
    ((21, 13, 32, 2), (3, 3, 32, 63), (1, 1), (1, 1), (1, 1)),     # 64 x 64, 273-pixel planes
    ((64, 67, 16, 4), (3, 3, 16, 63), (1, 1), (1, 1), (1, 1)),     # 64 x 128
    ((64, 65, 16, 4), (3, 3, 16, 127), (1, 1), (1, 1), (1, 1)),    # 128 x 128
    ((129, 127, 16, 1), (3, 3, 16, 129), (1, 1), (1, 1), (1, 1)),  # odd planes
    ((131, 129, 70, 2), (3, 3, 70, 16), (2, 2), (1, 1), (1, 1)),   # data gradient by phases
]


@pytest.mark.parametrize("out", ["f32", "t"])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("g", STORES, ids=lambda g: "x{}_w{}_s{}".format(*["x".join(map(str, v)) for v in g[:3]]))
def test_unsplit_results(af, rng, g, dt, out, monkeypatch):
    """The same bits as the element gather, which stores from registers."""
    t = {"bf16": af.bf16, "f16": af.f16}[dt]
    ot = af.f32 if out == "f32" else t
    X = af.Array(rng.standard_normal(g[0]).astype(np.float32)).astype(t)
    W = af.Array((rng.standard_normal(g[1]) * 0.1).astype(np.float32)).astype(t)
    monkeypatch.setenv("AFHIP_NN_GATHER", "1")
    monkeypatch.setenv("AFHIP_NN_SPLIT", "1")
    y = af.convolve2NN(X, W, *g[2:], out_type=ot)
    DY = af.Array(np.random.default_rng(7).standard_normal(y.dims).astype(np.float32)).astype(t)

    def both():
        y = af.convolve2NN(X, W, *g[2:], out_type=ot)
        dx = af.convolve2GradientNN(DY, X, W, y, *g[2:], af.AF_CONV_GRADIENT_DATA, out_type=ot)
        return y.astype(af.f32).to_numpy(), dx.astype(af.f32).to_numpy()

    got = both()
    monkeypatch.setenv("AFHIP_NN_CL", "0")
    for a, b in zip(got, both()):
        np.testing.assert_array_equal(a, b)
