// af_canny's kernels (kernels/canny_tiles.hip) as the dispatch calls them;
// return codes as in include/afhip_kernels.h.
#pragma once
#include <hip/hip_runtime.h>

namespace afhip {

// The largest suppressed value as n values whose maximum it is.
struct CannyMax {
    const float *v;
    int n;
};

// Smoothing, gradients and suppression of ns slices of d0 x d1 values of
// `dtype` into sup. part: canny_part_floats floats of scratch, which *top
// points into; one: *top is a single value.
long long canny_part_floats(long long d0, long long d1, long long ns);
int canny_suppress(int dtype, float *sup, CannyMax *top, float *part, const void *in, long long d0, long long d1,
                   long long ns, bool is_fast, bool one, hipStream_t s);

// Per slice the histogram of nbins over [0, maxval] into hist (cleared here).
int canny_histogram(unsigned *hist, const float *sup, long long per, long long ns, int nbins, float maxval,
                    hipStream_t s);
// Otsu's threshold (a bin index) per slice; _lanes: a lane per slice, any
// number of bins.
int canny_otsu_lanes(float *thr, const unsigned *hist, long long per, long long ns, int nbins, hipStream_t s);
int canny_otsu_bins(float *thr, const unsigned *hist, long long per, long long ns, int nbins, hipStream_t s);

// Thresholds and edge tracking. thr == nullptr: MANUAL, values over the
// largest against t1 and t2; otherwise against thr[slice] * t1 and thr[slice].
// labels: one unsigned per pixel of scratch.
int canny_track(unsigned char *out, unsigned *labels, const float *sup, CannyMax top, const float *thr, long long d0,
                long long d1, long long ns, float t1, float t2, hipStream_t s);

}  // namespace afhip
