// FP32 forward and data gradient on the BF16 matrix cores, three bfloat16
// parts per operand (kernels/nn.hip); arguments as afhip_k_conv2_nn_gemm_split
// (include/afhip_kernels.h) for f32 arrays at their own precision.
#pragma once
#include <hip/hip_runtime.h>

namespace afhip {

// Workspace bytes, 0 where the geometry is not served.
long long nn_x3_workspace(int pass, const long long *xdims, const long long *wdims, const long long *ydims,
                          const long long *stride, const long long *pad, const long long *dil, int nsplit);
int nn_x3(int pass, void *out, const void *in, const void *w, const long long *xdims, const long long *wdims,
          const long long *ydims, const long long *stride, const long long *pad, const long long *dil, int nsplit,
          void *workspace, long long workspace_bytes, hipStream_t s);

}  // namespace afhip
