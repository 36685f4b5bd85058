"""NN layers on a device with little memory left: where the copies that a GEMM
reads do not fit, the kernels that do without them run, with their bits."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _fill_device(L, leave):
    """Takes all but `leave` bytes of the device's memory; returns the blocks."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    blocks = []
    size = 1 << 60
    while True:
        assert L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        size = min(size, free.value - leave)
        if size < 8 * MB:
            return blocks
        p = ctypes.c_void_p()
        if L.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
            blocks.append(p)
        else:
            L.hipGetLastError()
            size //= 2


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_copies_that_do_not_fit(af, dt, monkeypatch):
    L, t = af.lib(), {"f32": af.f32, "bf16": af.bf16}[dt]
    # rows of 28 16-bit pixels and an FP32 3x3: the GEMMs, by rule
    dims, w = ((112, 112, 64, 32), (3, 3, 64, 64)) if dt == "f32" else ((28, 28, 128, 512), (3, 3, 128, 128))
    rng = np.random.default_rng(20261216)
    X = af.Array(rng.standard_normal(dims[::-1], dtype=np.float32).T).astype(t)
    DY = af.Array(rng.standard_normal(dims[::-1], dtype=np.float32).T).astype(t)
    W = af.Array(rng.standard_normal(w, dtype=np.float32)).astype(t)
    geo = ((1, 1), (1, 1), (1, 1))

    def step():
        for call in (lambda: af.convolve2NN(X, W, *geo),
                     lambda: af.convolve2GradientNN(DY, X, W, DY, *geo, af.AF_CONV_GRADIENT_DATA),
                     lambda: af.convolve2GradientNN(DY, X, W, DY, *geo, af.AF_CONV_GRADIENT_FILTER)):
            yield call().to_numpy()

    for name, value in (("AFHIP_NN_SMALL", "0"), ("AFHIP_NN_X3", "0"), ("AFHIP_NN_WG", "0")):
        monkeypatch.setenv(name, value)
    ref = list(step())
    for name in ("AFHIP_NN_SMALL", "AFHIP_NN_X3", "AFHIP_NN_WG"):
        monkeypatch.delenv(name)
    af.sync()
    assert L.af_device_gc() == 0
    # room for a result (103 MB) and not for a copy (154 MB in parts, 103 MB) beside it
    blocks = _fill_device(L, 170 * MB)
    try:
        for got, want in zip(step(), ref):
            np.testing.assert_array_equal(got, want)
            assert L.af_device_gc() == 0
    finally:
        for p in blocks:
            L.hipFree(p)
