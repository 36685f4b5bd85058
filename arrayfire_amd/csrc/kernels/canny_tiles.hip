// af_canny in tiles: the whole pipeline of src/api/c/canny.cpp:198-285 in four
// launches (five with many tiles; two more for AUTO_OTSU).
//
//  * canny_suppress_tile: conversion to float, the 5-tap separable smoothing,
//    Sobel, magnitude and non-maximum suppression of a 64 x 16 tile, each step
//    in LDS with the halo the next one needs, and the tile's largest value.
//    Every product and sum is rounded as in the separate steps (smoothing in
//    the order of src/backend/cpu/kernel/convolve.hpp:213-289 with its float
//    temp), so the map is the same to the bit. The image is read once and the
//    map written once where the separate kernels moved eight arrays; the halo
//    makes each tile compute 1.6 times its pixels in the smoothing.
//  * canny_label_tile, canny_label_borders, canny_label_out: edge tracking. The
//    marked set is the closure of the seeds over weak pixels: the weak pixels
//    whose connected component, in the graph of weak pixels and seeds under the
//    reference's eight linear-offset neighbours, holds a seed. Components are
//    found by union-find on labels (pixel index + 1; the parent of a label is
//    never larger), first inside a tile in LDS, then across tile borders with
//    device-scope atomics; every seed starts with label 0, so a component with
//    a seed has root 0 and needs no second pass. Three launches whatever the
//    shape of the edges, where sweeps over the image needed one launch per
//    pixel of the longest chain and a host read every 16 (96 launches and six
//    reads for a 1024^2 picture).
//
// 1024^2 f32, MANUAL: 39 us (suppression 13, labels in tiles 15, across tiles 8,
// out 5) against 666 to 930 us; each launch is one round of 1024 workgroups and
// bound by latency: the LDS steps of a tile, then chains of label reads.
#include <algorithm>

#include "kcommon.hpp"
#include "../canny.hpp"
#include "../../../include/afhip_kernels.h"

namespace afhip {

constexpr int CT_W = 64, CT_H = 16;  // tile: dim0 x dim1
constexpr int CT_N = CT_W * CT_H;
constexpr unsigned CT_NONE = 0xffffffffu;  // neither weak nor a seed

// cannyHelper's smoothing taps (src/api/c/canny.cpp:203-206)
__device__ constexpr float kCannyTap[5] = {-0.11021f, -0.23691f, -0.30576f, -0.23691f, -0.11021f};

__device__ inline int mirror101(int idx, int end) { return abs(end - abs(end - idx)); }

// e / W for a tile's indexes: one 24-bit product, where the general division
// by a constant takes two quarter-rate ones.
template <int W>
__host__ __device__ constexpr int tile_row(int e) {
    return (int)(((unsigned)e * ((1u << 18) / W + 1)) >> 18);
}
template <int W, int N>
constexpr bool tile_row_holds() {
    for (int e = 0; e < N; ++e)
        if (tile_row<W>(e) != e / W || (unsigned)e * ((1u << 18) / W + 1) >= (1u << 24)) return false;
    return true;
}

// The largest of the workgroup's 256 values (all >= 0), in every lane.
__device__ inline float block_max(float v) {
    __shared__ float red[4];
#pragma unroll
    for (int d = 32; d; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// Tile and slice of a workgroup, `first` being the launch's first tile;
// neighbouring tiles on one XCD share halo lines.
struct CannyTile {
    long long slice;
    int i0, j0;
};
__device__ inline CannyTile canny_tile(int d0, int d1, long long first) {
    const int nx = (d0 + CT_W - 1) / CT_W, ny = (d1 + CT_H - 1) / CT_H;
    const long long b = first + xcd_remap(blockIdx.x, gridDim.x);
    const int per = nx * ny;
    CannyTile t;
    t.slice = b / per;
    const int r = (int)(b - t.slice * per);
    t.i0 = r % nx * CT_W;
    t.j0 = r / nx * CT_H;
    return t;
}

template <typename T>
__global__ __launch_bounds__(256) void canny_suppress_tile(float *__restrict__ sup, float *__restrict__ part,
                                                           const T *__restrict__ in, int d0, int d1, int is_fast,
                                                           long long first) {
#pragma clang fp contract(off)
    constexpr int XW = CT_W + 8, XH = CT_H + 8;  // input: +-4
    constexpr int TW = CT_W + 4, TH = CT_H + 8;  // after the dim0 pass: +-2, +-4
    constexpr int SW = CT_W + 4, SH = CT_H + 4;  // smoothed: +-2
    constexpr int MW = CT_W + 2, MH = CT_H + 2;  // magnitude: +-1
    __shared__ float x[XH * XW], tmp[TH * TW], sm[SH * SW], mag[MH * MW];
    const CannyTile tl = canny_tile(d0, d1, first);
    const int i0 = tl.i0, j0 = tl.j0;
    const T *img = in + tl.slice * ((long long)d0 * d1);
    static_assert(tile_row_holds<XW, XW * XH + 256>() && tile_row_holds<TW, TW * TH>() && tile_row_holds<MW, MW * MH>());
    // pixels outside the image read as 0, as the convolution's DEFAULT border
    constexpr int NX = (XH * XW + 255) / 256;
    T v[NX];
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        const int e = (int)threadIdx.x + 256 * u, row = tile_row<XW>(e);
        const int i = min(max(i0 - 4 + e - row * XW, 0), d0 - 1), j = min(max(j0 - 4 + row, 0), d1 - 1);
        v[u] = img[j * d0 + i];
    }
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        const int e = (int)threadIdx.x + 256 * u, row = tile_row<XW>(e);
        const int i = i0 - 4 + e - row * XW, j = j0 - 4 + row;
        if (e < XH * XW) x[e] = i >= 0 && i < d0 && j >= 0 && j < d1 ? (float)v[u] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < (TH * TW + 255) / 256; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        if (e >= TH * TW) break;
        const float *p = x + e + tile_row<TW>(e) * (XW - TW) + 4;
        float acc = 0.f;
#pragma unroll
        for (int f = 0; f < 5; ++f) acc += p[-f] * kCannyTap[f];
        tmp[e] = acc;
    }
    __syncthreads();
    // the temp's rows outside the image are 0: their products add nothing
#pragma unroll
    for (int u = 0; u < (SH * SW + 255) / 256; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        if (e >= SH * SW) break;
        const float *p = tmp + e + 4 * TW;
        float acc = 0.f;
#pragma unroll
        for (int f = 0; f < 5; ++f) acc += p[-f * TW] * kCannyTap[f];
        sm[e] = acc;
    }
    __syncthreads();
    auto sobel = [&](int i, int j, float &dx, float &dy) {
        const int im = mirror101(i - 1, d0 - 1) - (i0 - 2), ip = mirror101(i + 1, d0 - 1) - (i0 - 2);
        const int jm = (mirror101(j - 1, d1 - 1) - (j0 - 2)) * SW, jp = (mirror101(j + 1, d1 - 1) - (j0 - 2)) * SW;
        const int ic = i - (i0 - 2), jc = (j - (j0 - 2)) * SW;
        const float NW = sm[jm + im], SWv = sm[jm + ip], NE = sm[jp + im], SE = sm[jp + ip];
        const float N = sm[jc + im], S = sm[jc + ip], W = sm[jm + ic], E = sm[jp + ic];
        dx = ((SWv + SE) - (NW + NE)) + 2.0f * (S - N);
        dy = ((NE + SE) - (NW + SWv)) + 2.0f * (E - W);
    };
#pragma unroll
    for (int u = 0; u < (MH * MW + 255) / 256; ++u) {
        const int e = (int)threadIdx.x + 256 * u, row = tile_row<MW>(e);
        if (e >= MH * MW) break;
        const int i = i0 - 1 + e - row * MW, j = j0 - 1 + row;
        float m = 0.f;
        if (i >= 0 && i < d0 && j >= 0 && j < d1) {
            float dx, dy;
            sobel(i, j, dx, dy);
            m = is_fast ? fabsf(dx) + fabsf(dy) : sqrtf(dx * dx + dy * dy);
        }
        mag[e] = m;
    }
    __syncthreads();
    float top = 0.f;
#pragma unroll
    for (int q = 0; q < CT_N / 256; ++q) {
        const int e = (int)threadIdx.x + 256 * q, i = i0 + e % CT_W, j = j0 + e / CT_W;
        if (i >= d0 || j >= d1) continue;
        float res = 0.f;
        if (i >= 1 && i < d0 - 1 && j >= 1 && j < d1 - 1) {
            const float *m = mag + (e / CT_W + 1) * MW + e % CT_W + 1;
            const float curr = m[0];
            if (curr != 0.f) {
                const float se = m[MW + 1], nw = m[-MW - 1], ea = m[1], we = m[-1];
                const float ne = m[-MW + 1], sw = m[MW - 1], no = m[-MW], so = m[MW];
                float dx, dy;
                sobel(i, j, dx, dy);
                // the neighbours on either side of the gradient's direction, and
                // its share of the diagonal ones: the smaller over the larger
                // derivative (one division for the four quadrants)
                const bool px = dx >= 0, py = dy >= 0;
                const bool g = (px ? (py ? dx - dy : dx + dy) : (py ? dx + dy : -dx + dy)) >= 0;
                // quadrants (+,+) and (+,-): g picks dim0; (-,+): g picks dim1; (-,-): dim0
                const bool along0 = (px || !py) ? g : !g;
                const bool fwd0 = px, fwd1 = py;
                const float a1 = along0 ? (fwd0 ? ea : we) : (fwd1 ? so : no);
                const float a2 = along0 ? (fwd0 ? we : ea) : (fwd1 ? no : so);
                const float b1 = px ? (py ? se : ne) : (py ? sw : nw);
                const float b2 = px ? (py ? nw : sw) : (py ? ne : se);
                const float num = along0 ? dy : dx, den = along0 ? dx : dy;
                const float alpha = (px == py ? num : -num) / den;
                const float mag1 = (1.0f - alpha) * a1 + alpha * b1;
                const float mag2 = (1.0f - alpha) * a2 + alpha * b2;
                if (curr > mag1 && curr > mag2) res = curr;
            }
        }
        sup[tl.slice * ((long long)d0 * d1) + (long long)j * d0 + i] = res;
        top = fmaxf(top, res);
    }
    top = block_max(top);
    if (threadIdx.x == 0) part[first + blockIdx.x] = top;
}

// A value per workgroup: the largest of its share of part.
__global__ __launch_bounds__(256) void canny_max_final(float *__restrict__ out, const float *__restrict__ part,
                                                       long long n) {
    float v = 0.f;
    for (long long e = blockIdx.x * 256LL + threadIdx.x; e < n; e += gridDim.x * 256LL) v = fmaxf(v, part[e]);
    v = block_max(v);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// hist [ns][nbins]: bin = (int)(v / step) clamped to [0, nbins-1]. Counts are
// kept in LDS per workgroup, which has one slice's share, up to CH_BINS bins;
// most pixels are suppressed to 0 and share one bin, which device atomics
// would take one at a time.
constexpr int CH_BINS = 8192;
__global__ __launch_bounds__(256) void canny_hist_tile(unsigned *__restrict__ hist, const float *__restrict__ v,
                                                       long long per, int blocks_per_slice, int nbins, float step,
                                                       long long first) {
#pragma clang fp contract(off)
    extern __shared__ unsigned bins[];
    const long long b = first + blockIdx.x, sl = b / blocks_per_slice;
    const int part = (int)(b - sl * blocks_per_slice);
    const bool lds = nbins <= CH_BINS;
    if (lds) {
        for (int b = threadIdx.x; b < nbins; b += 256) bins[b] = 0;
        __syncthreads();
    }
    unsigned zeros = 0;
    for (long long e = part * 256LL + threadIdx.x; e < per; e += blocks_per_slice * 256LL) {
        int b = (int)((v[sl * per + e] - 0.0f) / step);
        b = max(b, 0);
        b = min(b, nbins - 1);
        if (b == 0) ++zeros;
        else if (lds) atomicAdd(bins + b, 1u);
        else atomicAdd(hist + sl * nbins + b, 1u);
    }
#pragma unroll
    for (int d = 32; d; d >>= 1) zeros += __shfl_xor(zeros, d);
    if ((threadIdx.x & 63) == 0 && zeros) atomicAdd(lds ? bins : hist + sl * nbins, zeros);
    if (lds) {
        __syncthreads();
        for (int b = threadIdx.x; b < nbins; b += 256)
            if (bins[b]) atomicAdd(hist + sl * nbins + b, bins[b]);
    }
}

// Otsu's threshold per slice (src/api/c/canny.cpp:82-147) as canny_otsu: the
// sums over the bins run in bin order in one lane each (the class weight in
// the first wave, the class mean's sum in the second; the total's mean is that
// sum after the last bin), everything else in all lanes. 700 bins: 81 us in
// one lane, with its divisions in the chain.
constexpr int CO_BINS = 4096;
__global__ __launch_bounds__(256) void canny_otsu_slice(float *__restrict__ thr, const unsigned *__restrict__ hist,
                                                        int nbins, float total, long long first) {
#pragma clang fp contract(off)
    __shared__ float w[CO_BINS], m[CO_BINS];
    __shared__ float bk[4];
    __shared__ int bi[4];
    const unsigned *h = hist + (first + blockIdx.x) * nbins;
    const int t = threadIdx.x;
    for (int b = t; b < nbins; b += 256) {
        const float f = (float)h[b] / total;
        w[b] = f;
        m[b] = (float)b * f;
    }
    __syncthreads();
    if (t == 0 || t == 64) {
        float *p = t ? m : w, c = 0.f;
        int b = 0;
        for (; b + 8 <= nbins; b += 8) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = p[b + k];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                c = c + v[k];
                p[b + k] = c;
            }
        }
        for (; b < nbins; ++b) {
            c = c + p[b];
            p[b] = c;
        }
    }
    __syncthreads();
    const float ws = m[nbins - 1];
    // the first largest |sigma|; a NaN in bin 0 counts as the lowest float, a
    // later one never wins
    float best = -2.f;
    int at = 0;
    for (int b = t; b < nbins - 1; b += 256) {
        const float qL = w[b], cprod = m[b];
        const float qH = 1.0f - qL;
        const float muL = cprod / qL;
        const float muH = (ws - cprod) / qH;
        const float diff = muL - muH;
        const float sig = (diff * diff) * (qL * qH);
        const float key = sig != sig ? (b == 0 ? 3.402823466e38f : -1.f) : fabsf(sig);
        if (key > best) {
            best = key;
            at = b;
        }
    }
    auto take = [&](float k, int i) {
        if (k > best || (k == best && i < at)) {
            best = k;
            at = i;
        }
    };
#pragma unroll
    for (int d = 32; d; d >>= 1) {
        const float k = __shfl_xor(best, d);
        const int i = __shfl_xor(at, d);
        take(k, i);
    }
    if ((t & 63) == 0) {
        bk[t >> 6] = best;
        bi[t >> 6] = at;
    }
    __syncthreads();
    if (t == 0) {
        for (int k = 1; k < 4; ++k) take(bk[k], bi[k]);
        thr[first + blockIdx.x] = (float)at;
    }
}

__global__ __launch_bounds__(256) void canny_zero(unsigned *__restrict__ p, long long n) {
    for (long long e = blockIdx.x * 256LL + threadIdx.x; e < n; e += gridDim.x * 256LL) p[e] = 0;
}

// Union-find over labels x >= 1 with parent(x) = L[x - 1] <= x and the shared
// root 0. Parents only decrease, so every walk ends, and a walk that reads an
// older parent still ends in the same component.
struct LdsLabels {
    unsigned *L;
    __device__ unsigned parent(unsigned x) const { return *(volatile unsigned *)(L + x - 1); }
    __device__ unsigned lower(unsigned x, unsigned to) const { return atomicMin(L + x - 1, to); }
};
struct DeviceLabels {
    unsigned *L;
    __device__ unsigned parent(unsigned x) const {
        return __hip_atomic_load(L + x - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ unsigned lower(unsigned x, unsigned to) const {
        return __hip_atomic_fetch_min(L + x - 1, to, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
template <typename S>
__device__ inline unsigned label_root(const S &s, unsigned x) {
    while (x) {
        const unsigned y = s.parent(x);
        if (y == x) break;
        x = y;
    }
    return x;
}
template <typename S>
__device__ inline void label_join(const S &s, unsigned a, unsigned b) {
    for (;;) {
        a = label_root(s, a);
        b = label_root(s, b);
        if (a == b) return;
        if (a < b) {
            const unsigned c = a;
            a = b;
            b = c;
        }
        // a was a root when it was read; if it has been joined since, what it
        // was joined to (smaller than a) is joined to b in the next turn
        const unsigned was = s.lower(a, b);
        if (was == a) return;
        a = was;
    }
}

__global__ __launch_bounds__(256) void canny_label_tile(unsigned *__restrict__ labels, const float *__restrict__ sup,
                                                        const float *__restrict__ maxv, int nmax,
                                                        const float *__restrict__ thr, int d0, int d1, float t1,
                                                        float t2, long long first) {
#pragma clang fp contract(off)
    __shared__ unsigned L[CT_N];
    __shared__ unsigned long long mask[CT_H];
    const CannyTile tl = canny_tile(d0, d1, first);
    const long long per = (long long)d0 * d1;
    const long long base = tl.slice * per;
    const long long s0 = d0 + 1, s1 = s0 + (long long)(d0 - 1) * (d1 - 1);  // the reference's seed scan
    const int col = threadIdx.x & 63;
    // the pixels' loads are in flight while the largest value is reduced
    float val[CT_N / 256];
#pragma unroll
    for (int q = 0; q < CT_N / 256; ++q) {
        const int i = min(tl.i0 + col, d0 - 1), j = min(tl.j0 + ((int)threadIdx.x >> 6) + 4 * q, d1 - 1);
        val[q] = sup[base + j * d0 + i];
    }
    float T1 = t1, T2 = t2, den = 1.f;
    if (thr) {
        T2 = thr[tl.slice];
        T1 = T2 * t1;
    } else {
        float m = 0.f;
        for (int e = threadIdx.x; e < nmax; e += 256) m = fmaxf(m, maxv[e]);
        den = block_max(m);  // the map's minimum is 0: its borders are suppressed
    }
    // A wave holds a row of the tile. Runs along the row join without atomics:
    // every pixel of a run starts below the run's first pixel, or below 0 when
    // the run holds a seed.
    static_assert(CT_W == 64, "a row is a wave");
    unsigned long long mine[CT_N / 256];
#pragma unroll
    for (int q = 0; q < CT_N / 256; ++q) {
        const int row = ((int)threadIdx.x >> 6) + 4 * q, i = tl.i0 + col, j = tl.j0 + row;
        bool weak = false, seed = false;
        if (i < d0 && j < d1) {
            const long long r = (long long)j * d0 + i;
            const float g = thr ? val[q] : val[q] / den;
            seed = g >= T2 && r >= s0 && r < s1;
            weak = !(g >= T2) && g >= T1;
        }
        const unsigned long long f = __ballot(weak || seed), sd = __ballot(seed);
        mine[q] = f;
        if (col == 0) mask[row] = f;
        unsigned l = CT_NONE;
        if (f >> col & 1) {
            const unsigned long long gaps = ~f;
            const unsigned long long below = gaps & ((1ull << col) - 1), above = gaps & (~0ull << col);
            const int first = below ? 64 - __clzll((long long)below) : 0;
            const int end = above ? __ffsll((long long)above) - 1 : 64;  // past the run
            const unsigned long long run = (end == 64 ? ~0ull : (1ull << end) - 1) & (~0ull << first);
            l = sd & run ? 0 : (unsigned)(row * CT_W + first) + 1;
        }
        L[row * CT_W + col] = l;
    }
    __syncthreads();
    const LdsLabels S{L};
    // Between rows one join per contact of two runs is enough: with the pixel
    // above when the pair to the left is not one already, with a diagonal one
    // when neither the pixel above nor the neighbour on that side is there.
#pragma unroll
    for (int q = 0; q < CT_N / 256; ++q) {
        const int row = ((int)threadIdx.x >> 6) + 4 * q, e = row * CT_W + col;
        if (row == 0) continue;
        const unsigned long long f = mine[q], u = mask[row - 1], bit = 1ull << col;
        if (f & u & ~(f << 1 & u << 1) & bit) label_join(S, e + 1, e - CT_W + 1);
        if (f & u << 1 & ~u & ~(f << 1) & bit) label_join(S, e + 1, e - CT_W);
        if (f & u >> 1 & ~u & ~(f >> 1) & bit) label_join(S, e + 1, e - CT_W + 2);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < CT_N / 256; ++q) {
        const int e = (int)threadIdx.x + 256 * q, i = tl.i0 + e % CT_W, j = tl.j0 + e / CT_W;
        if (i >= d0 || j >= d1) continue;
        unsigned l = CT_NONE;
        if (mine[q] >> col & 1) {
            const unsigned r = label_root(S, e + 1);
            l = r == 0 ? 0 : (unsigned)((tl.j0 + (int)(r - 1) / CT_W) * d0 + tl.i0 + (int)(r - 1) % CT_W) + 1;
        }
        labels[base + (long long)j * d0 + i] = l;
    }
}

// Joins across tile borders. Lanes 0..63 take the tile's first row, the next
// 2 x 16 its first and last columns: those pixels hold every pair of linear
// neighbours (the smaller index second) that canny_label_tile has not joined,
// the pairs that wrap from one column of the image to the next included.
__global__ __launch_bounds__(128) void canny_label_borders(unsigned *__restrict__ labels, int d0, int d1,
                                                           long long first) {
    const CannyTile tl = canny_tile(d0, d1, first);
    const int t = threadIdx.x;
    int i, j;
    if (t < CT_W) {
        i = tl.i0 + t;
        j = tl.j0;
    } else if (t < CT_W + 2 * CT_H) {
        i = t < CT_W + CT_H ? tl.i0 : min(tl.i0 + CT_W, d0) - 1;
        j = tl.j0 + (t - CT_W) % CT_H;
    } else {
        return;
    }
    if (i >= d0 || j >= d1) return;
    const DeviceLabels S{labels + tl.slice * ((long long)d0 * d1)};
    const int r = j * d0 + i;
    const int off[4] = {-1, -d0 - 1, -d0, -d0 + 1};
    // all five labels in flight at once; a join starts from the parents read
    const unsigned own = S.parent(r + 1);
    unsigned l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) l[k] = S.parent(max(r + off[k], 0) + 1);
    if (own == CT_NONE) return;
    unsigned last = own;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int q = r + off[k];
        if (q < 0 || l[k] == CT_NONE || l[k] == last) continue;
        const int qi = q % d0, qj = q / d0;
        if (qi / CT_W == i / CT_W && qj / CT_H == j / CT_H && abs(qi - i) <= 1) continue;
        last = l[k];
        label_join(S, own, last);
    }
}

__global__ __launch_bounds__(256) void canny_label_out(unsigned char *__restrict__ out,
                                                       const unsigned *__restrict__ labels, long long per,
                                                       long long n) {
    for (long long e = blockIdx.x * 256LL + threadIdx.x; e < n; e += gridDim.x * 256LL) {
        unsigned x = labels[e];
        unsigned char o = 0;
        if (x != CT_NONE) {
            const unsigned *L = labels + e / per * per;
            unsigned y;
            while (x && (y = L[x - 1]) != x) x = y;
            o = x == 0;
        }
        out[e] = o;
    }
}

static long long canny_tiles(long long d0, long long d1, long long ns) {
    return (d0 + CT_W - 1) / CT_W * ((d1 + CT_H - 1) / CT_H) * ns;
}

// The tile maxima, then one value or up to 1024.
constexpr int CT_MAXIMA = 1024;
long long canny_part_floats(long long d0, long long d1, long long ns) { return canny_tiles(d0, d1, ns) + 1 + CT_MAXIMA; }

// Launches of n workgroups, as many at a time as one launch takes (a batch of
// very many small images, or an image a few pixels wide, has more tiles).
template <typename Fn>
static void canny_launches(long long n, Fn launch) {
    for (long long first = 0; first < n; first += kMaxGrid256)
        launch((unsigned)std::min(n - first, kMaxGrid256), first);
}

template <typename T>
static void launch_suppress(float *sup, float *part, const void *in, long long d0, long long d1, long long tiles,
                            bool is_fast, hipStream_t s) {
    canny_launches(tiles, [&](unsigned nb, long long first) {
        canny_suppress_tile<T><<<nb, 256, 0, s>>>(sup, part, (const T *)in, (int)d0, (int)d1, is_fast, first);
    });
}

int canny_suppress(int dtype, float *sup, CannyMax *top, float *part, const void *in, long long d0, long long d1,
                   long long ns, bool is_fast, bool one, hipStream_t s) {
    const long long tiles = canny_tiles(d0, d1, ns);
    if (d0 < 2 || d1 < 2 || d0 * d1 >= (1LL << 31)) return K_ERR_SIZE;
    switch (dtype) {
        case DT_F32: launch_suppress<float>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_F64: launch_suppress<double>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_S32: launch_suppress<int32_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_U32: launch_suppress<uint32_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_S16: launch_suppress<int16_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_U16: launch_suppress<uint16_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_S8: launch_suppress<int8_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        case DT_U8: launch_suppress<uint8_t>(sup, part, in, d0, d1, tiles, is_fast, s); break;
        default: return K_ERR_TYPE;
    }
    // the tile kernel of canny_track reduces up to 1024 values itself, which
    // costs each workgroup four loads per lane and saves the launch
    const float *v = part;
    long long n = tiles;
    if (n > 64 * 4 * CT_MAXIMA) {  // too many for one workgroup
        float *few = part + tiles + 1;
        canny_max_final<<<CT_MAXIMA, 256, 0, s>>>(few, v, n);
        v = few;
        n = CT_MAXIMA;
    }
    if (one || n > CT_MAXIMA) {
        canny_max_final<<<1, 256, 0, s>>>(part + tiles, v, n);
        v = part + tiles;
        n = 1;
    }
    top->v = v;
    top->n = (int)n;
    return launch_status();
}

int canny_histogram(unsigned *hist, const float *sup, long long per, long long ns, int nbins, float maxval,
                    hipStream_t s) {
    if (nbins < 1) return K_ERR_ARG;
    const float step = (float)(((double)maxval - 0.0) / (double)(float)nbins);
    const long long nz = (long long)nbins * ns;
    canny_zero<<<(unsigned)std::min<long long>((nz + 255) / 256, kMaxGridBlocks), 256, 0, s>>>(hist, nz);
    // about 16 values per lane, at most 256 workgroups per slice
    const int bps = (int)std::min<long long>((per + 4095) / 4096, 256);
    canny_launches(ns * bps, [&](unsigned nb, long long first) {
        canny_hist_tile<<<nb, 256, nbins <= CH_BINS ? nbins * sizeof(unsigned) : 0, s>>>(hist, sup, per, bps, nbins,
                                                                                        step, first);
    });
    return launch_status();
}

// One workgroup per slice up to CO_BINS bins (two LDS arrays), one lane per
// slice past them.
int canny_otsu_bins(float *thr, const unsigned *hist, long long per, long long ns, int nbins, hipStream_t s) {
    if (nbins > CO_BINS) return canny_otsu_lanes(thr, hist, per, ns, nbins, s);
    canny_launches(ns, [&](unsigned nb, long long first) {
        canny_otsu_slice<<<nb, 256, 0, s>>>(thr, hist, nbins, (float)per, first);
    });
    return launch_status();
}

int canny_track(unsigned char *out, unsigned *labels, const float *sup, CannyMax top, const float *thr,
                long long d0, long long d1, long long ns, float t1, float t2, hipStream_t s) {
    const long long tiles = canny_tiles(d0, d1, ns), n = d0 * d1 * ns;
    canny_launches(tiles, [&](unsigned nb, long long first) {
        canny_label_tile<<<nb, 256, 0, s>>>(labels, sup, top.v, top.n, thr, (int)d0, (int)d1, t1, t2, first);
    });
    canny_launches(tiles, [&](unsigned nb, long long first) {
        canny_label_borders<<<nb, 128, 0, s>>>(labels, (int)d0, (int)d1, first);
    });
    canny_label_out<<<(unsigned)std::min<long long>((n + 255) / 256, kMaxGridBlocks), 256, 0, s>>>(out, labels,
                                                                                                  d0 * d1, n);
    return launch_status();
}

}  // namespace afhip
