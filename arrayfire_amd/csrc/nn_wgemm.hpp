// Filter gradient from channel-last copies (kernels/nn_wgemm.hip), any
// geometry: bf16 and f16 arrays at their own precision, f32 arrays in three
// BF16 parts per operand. type: af_dtype of x and dy; cus: compute units
// (the split of the pixels follows from it).
#pragma once
#include <hip/hip_runtime.h>

namespace afhip {

// Workspace bytes, 0 where not served.
long long nn_wgemm_workspace(int type, const long long *xdims, const long long *wdims, const long long *ydims,
                             const long long *stride, const long long *pad, const long long *dil, int cus);
int nn_wgemm(int type, int out_type, void *dw, const void *x, const void *dy, const long long *xdims,
             const long long *wdims, const long long *ydims, const long long *stride, const long long *pad,
             const long long *dil, int cus, void *workspace, long long workspace_bytes, hipStream_t s);

}  // namespace afhip
