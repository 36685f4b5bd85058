"""The Canny steps of the kernel ABI, one by one, against af_canny, whose tile
kernels run them fused: the same map exactly, for batches, both magnitudes and
both kinds of threshold."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _p(a, off=0):
    return ctypes.c_void_p(a.device_ptr() + off)


@pytest.mark.parametrize("otsu", [False, True], ids=["manual", "otsu"])
@pytest.mark.parametrize("fast", [0, 1], ids=["l2", "l1"])
@pytest.mark.parametrize("dims", [(5, 5), (70, 33), (130, 50, 3)], ids=lambda d: "x".join(map(str, d)))
def test_steps(af, rng, dims, fast, otsu):
    L, ll, f32 = af.lib(), ctypes.c_longlong, ctypes.c_float
    stream = ctypes.c_void_p(af.stream())
    lo, hi = (0.4, 0.0) if otsu else (0.1, 0.4)
    img = (rng.random(dims) * 200).astype(np.float32)
    d0, d1 = dims[:2]
    per, ns = d0 * d1, int(np.prod(dims[2:], dtype=int))
    n = per * ns
    X = af.Array(img)
    taps = af.Array(np.array([-0.11021, -0.23691, -0.30576, -0.23691, -0.11021], np.float32))
    tmp, smooth, gx, gy, mag, sup = (af.constant(0, (n,)) for _ in range(6))
    mm, part = af.constant(0, (2,)), af.constant(0, (2048,))
    strong, weak, out = (af.constant(0, (n,), af.u8) for _ in range(3))
    size = (ll * 4)(d0, d1, ns, 1)
    assert L.afhip_k_convolve2_sep(af.f32, _p(smooth), size, _p(X), size, _p(taps), ll(5), _p(taps), ll(5), 0, _p(tmp),
                                   stream) == 0
    assert L.afhip_k_canny_grad(_p(gx), _p(gy), _p(mag), _p(smooth), ll(d0), ll(d1), ll(ns), fast, stream) == 0
    assert L.afhip_k_canny_nms(_p(sup), _p(mag), _p(gx), _p(gy), ll(d0), ll(d1), ll(ns), stream) == 0
    assert L.afhip_k_canny_minmax(_p(mm), _p(sup), ll(n), _p(part), stream) == 0
    thr = None
    if otsu:
        top = float(mm.to_numpy().ravel()[1])
        bins, thr = af.constant(0, (int(top) * ns,), af.u32), af.constant(0, (ns,))
        assert L.afhip_k_canny_otsu(_p(thr), _p(bins), _p(sup), ll(per), ll(ns), int(top), f32(top), stream) == 0
    assert L.afhip_k_canny_candidates(_p(strong), _p(weak), _p(sup), _p(mm), _p(thr) if otsu else None, ll(per), ll(ns),
                                      f32(lo), f32(hi), int(otsu), stream) == 0
    assert L.afhip_k_canny_seed(_p(out), _p(strong), ll(d0), ll(d1), ll(ns), stream) == 0
    for _ in range(n):
        changed = af.constant(0, (1,), af.u32)
        assert L.afhip_k_canny_sweep(_p(out), _p(weak), ll(d0), ll(d1), ll(ns), _p(changed), stream) == 0
        if not changed.to_numpy().any():
            break
    ref = af.canny(img, int(otsu), lo, hi, 3, bool(fast)).to_numpy().astype(np.uint8)
    np.testing.assert_array_equal(out.to_numpy().ravel(), ref.ravel(order="F"))
    assert ref.any()
