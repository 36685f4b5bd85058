// af_canny (src/api/c/canny.cpp:198-285): the 5-tap separable smoothing of
// the convolution path, then Sobel gradients, non-maximum suppression,
// thresholds (MANUAL or AUTO_OTSU) and edge tracking by hysteresis, all on
// the GPU (kernels/canny_tiles.hip). The host reads one scalar (the suppressed
// map's maximum) for the Otsu bin count; MANUAL reads nothing.
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/af/array.h"
#include "../../include/af/image.h"
#include "canny.hpp"
#include "runtime.hpp"

namespace afhip {

static af_array canny(const ArrayImpl &in, af_canny_threshold ct, float t1, float t2, bool is_fast) {
    const dim4 d = in.dims;
    const dim_t d0 = d[0], d1 = d[1], ns = d[2] * d[3], n = d.elements();
    hipStream_t s = stream();
    const bool otsu = ct == AF_CANNY_THRESHOLD_AUTO_OTSU;
    auto sup = scratch(sizeof(float) * n), part = scratch(sizeof(float) * canny_part_floats(d0, d1, ns));
    CannyMax top;
    check_k(canny_suppress(in.type, (float *)sup->ptr, &top, (float *)part->ptr, in.data(), d0, d1, ns, is_fast, otsu,
                           s),
            "canny");
    std::shared_ptr<Buffer> thr;
    if (otsu) {
        float maxv = 0;
        check_hip(hipMemcpyAsync(&maxv, top.v, sizeof(maxv), hipMemcpyDeviceToHost, s), "canny");
        sync_stream();
        const unsigned nbins = static_cast<unsigned>(maxv);
        if (nbins < 1) AFHIP_THROW(AF_ERR_ARG, "canny: the gradient's maximum is below one Otsu bin");
        auto hist = scratch(sizeof(unsigned) * nbins * ns);
        check_k(canny_histogram((unsigned *)hist->ptr, (const float *)sup->ptr, d0 * d1, ns, (int)nbins, maxv, s),
                "canny");
        thr = scratch(sizeof(float) * ns);
        check_k(canny_otsu_bins((float *)thr->ptr, (const unsigned *)hist->ptr, d0 * d1, ns, (int)nbins, s), "canny");
    }
    auto labels = scratch(sizeof(unsigned) * n);
    NewHandle out(make_handle(b8, d));
    check_k(canny_track((unsigned char *)out.data(), (unsigned *)labels->ptr, (const float *)sup->ptr, top,
                        thr ? (const float *)thr->ptr : nullptr, d0, d1, ns, t1, t2, s),
            "canny");
    return out.release();
}

}  // namespace afhip

using namespace afhip;

// src/api/c/canny.cpp:224-285
AFAPI af_err af_canny(af_array *out, const af_array in, const af_canny_threshold ct, const float t1, const float t2,
                      const unsigned sw, const bool isf) {
    try {
        ARG_ASSERT(0, out != nullptr);
        const ArrayImpl &a = get(in);
        const dim4 dims = a.dims;
        DIM_ASSERT(2, dims.ndims() >= 2);
        DIM_ASSERT(2, dims[0] >= 5 && dims[1] >= 5);
        ARG_ASSERT(5, sw == 3);
        switch (a.type) {
            case f32:
            case f64:
            case s32:
            case u32:
            case s16:
            case u16:
            case s8:
            case u8: break;
            default: TYPE_ERROR(1, a.type);
        }
        DIM_ASSERT(1, dims[0] * dims[1] < (1LL << 31));
        *out = canny(a, ct, t1, t2, isf);
    }
    CATCHALL;
    return AF_SUCCESS;
}
