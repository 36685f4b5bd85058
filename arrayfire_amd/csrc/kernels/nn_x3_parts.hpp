// An FP32 value as the sum of three bfloat16 values, x = x1 + x2 + x3 (each the
// rounding of what the ones before leave), and the range in which that is
// exact to FP32's 24 bits: zeros and magnitudes 2^-100 .. 2^63, for which every
// part is a normal bfloat16 and no product of two values overflows.
#pragma once
#include "kcommon.hpp"

namespace afhip {

constexpr unsigned X3_LO = 27u << 23, X3_HI = 190u << 23;

__device__ __forceinline__ bool x3_odd_value(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v) & 0x7fffffffu;
    return u != 0 && u - X3_LO >= X3_HI - X3_LO;
}
__device__ __forceinline__ void x3_parts(float v, uint16_t (&h)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h[k] = f32_to_bf16_bits(v);
        v -= bf16_bits_to_f32(h[k]);
    }
}

// 64 pixels by one 32-channel slice of an NCHW array to the channel-last
// layout [pixel][slice][part][32], zeros past the Cd channels, by a 256-lane
// workgroup; block b counts slices first. Returns whether the lane saw a value
// outside the range.
__device__ __forceinline__ int x3_copy_block(uint16_t *__restrict__ dst, const float *__restrict__ src, int b, int hw,
                                             int Cd, int npix, int slices, unsigned (*tile)[64 * 17]) {
    const int pb = b / slices, cs = b - pb * slices;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int pix = min(pb * 64 + lane, npix - 1), n = pix / hw;
    const float *s = src + (long long)n * Cd * hw + (pix - n * hw);
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = s[(long long)min(cs * 32 + wave * 8 + u, Cd - 1) * hw];
    uint16_t h[8][3];
    int odd = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float x = cs * 32 + wave * 8 + u < Cd ? v[u] : 0.f;
        odd |= x3_odd_value(x);
        x3_parts(x, h[u]);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int u = 0; u < 8; u += 2) tile[q][lane * 17 + wave * 4 + u / 2] = h[u][q] | (unsigned)h[u + 1][q] << 16;
    __syncthreads();
    // 64 pixels x 3 parts x 4 groups of 16 bytes
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int e = (int)threadIdx.x + 256 * u, px = e / 12, g = e - px * 12;
        if (pb * 64 + px < npix) {
            const unsigned *q = tile[g >> 2] + px * 17 + (g & 3) * 4;
            *reinterpret_cast<uint4 *>(dst + ((long long)(pb * 64 + px) * slices + cs) * 96 + g * 8) =
                make_uint4(q[0], q[1], q[2], q[3]);
        }
    }
    return odd;
}

}  // namespace afhip
