// An FP32 value, times 2^16, as the sum of three bfloat16 values, x = x1 + x2 +
// x3 (each the rounding of what the ones before leave). That is exact to FP32's
// 24 bits for every magnitude below 2^32: the scale lifts the last place of the
// smallest denormal to the last place of bfloat16's (2^-133), and the matrix
// cores take and return denormals. Sums are formed of products scaled by 2^32
// and scaled back once; below 2^32 a sum of 2^28 of them stays under 2^124.
// What is left are values of 2^32 and more, infinities and NaNs.
#pragma once
#include "kcommon.hpp"

namespace afhip {

constexpr float X3_SCALE = 65536.f, X3_UNSCALE = 1.f / (65536.f * 65536.f);

// What a block of values holds, a bit each.
enum X3Flag : int {
    X3_HUGE = 1,   // magnitudes from 2^32, infinities, NaNs
    X3_TINY = 2,   // other than zero below 2^-100
    X3_PLAIN = 4,  // in between
};
__device__ __forceinline__ int x3_flag(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v) & 0x7fffffffu;
    return u >= 159u << 23 ? X3_HUGE : u >= 27u << 23 ? X3_PLAIN : u ? X3_TINY : 0;
}
// The flags of a 256-lane workgroup's values, in every lane; once per kernel.
__device__ __forceinline__ int x3_block_flags(int f) {
    __shared__ int wave[4];
    int b = 0;
#pragma unroll
    for (int k = 1; k <= X3_PLAIN; k *= 2) b |= __any(f & k) ? k : 0;
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = b;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(wave[0] | wave[1] | wave[2] | wave[3]);
}
constexpr uint16_t X3_RAW = 0x7fff;  // first part of a value stored as it is
__device__ __forceinline__ void x3_parts(float v, uint16_t (&h)[3]) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    v *= X3_SCALE;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        h[k] = f32_to_bf16_bits(v);
        v -= bf16_bits_to_f32(h[k]);
    }
    if (x3_flag(__builtin_bit_cast(float, u)) == X3_HUGE) {
        h[0] = X3_RAW;
        h[1] = (uint16_t)(u >> 16);
        h[2] = (uint16_t)u;
    }
}
__device__ __forceinline__ float x3_value(unsigned a, unsigned b, unsigned c) {  // 16 bits each
    const float v = ((bf16_bits_to_f32((uint16_t)a) + bf16_bits_to_f32((uint16_t)b)) + bf16_bits_to_f32((uint16_t)c)) *
                    (1.f / X3_SCALE);
    return a == X3_RAW ? __builtin_bit_cast(float, b << 16 | c) : v;
}

// 64 pixels by one 32-channel slice of an NCHW array to the channel-last
// layout [pixel][slice][part][32], zeros past the Cd channels, by a 256-lane
// workgroup; block b counts slices first. Returns the flags of the lane's values.
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
    int flag = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float x = cs * 32 + wave * 8 + u < Cd ? v[u] : 0.f;
        flag |= x3_flag(x);
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
    return flag;
}

}  // namespace afhip
