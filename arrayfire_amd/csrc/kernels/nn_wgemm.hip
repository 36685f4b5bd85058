// convolve2_nn filter gradient as a GEMM over channel-last copies:
//   dw[k][c][tap] = sum over output pixels q of dy[q][k] * x[pixel(q, tap)][c]
// (src/backend/cpu/convolve.cpp:213-243), for any filter, stride, padding and
// dilation. The reduction runs over pixels, which the channel-last layout has
// as rows: a workgroup stages 32-pixel slices of 64 channels of each operand in
// LDS by whole 128-byte rows, whatever the tap's shift does to the pixels, and
// the MFMA fragments, eight pixels of one channel per lane, come from LDS
// through the transposing read (ds_read_b64_tr_b16). Kernels that keep pixels
// innermost need the shifted rows realigned (nn_wgrad.hip, filter sides 1 and
// 3) or gather element by element (nn_gemm).
//
// Workgroup: 256 lanes, 64 filters x 64 channels x up to three taps, one split
// of the pixels; 2 x 2 waves of 32 x 32 per tap, the dy fragments shared by the
// taps. Splits write FP32 partial gradients [split][tap][k][c], which
// nn_wgemm_sum adds in split order.
//
// f32 arrays run in three BF16 parts per operand (nn_x3_parts.hpp): six part
// products, the small ones in accumulators of their own; a workgroup that reads
// a block with huge values puts the parts together again and multiplies in FP32.
//
// us for the call, copies and sum included, against the kernels it replaces or
// competes with (dims W H C N -> K): BF16 28x28x128x16 -> 128 3x3 stride 2: 17
// (37, rows of 14 unaligned pixels), 55x47x64x8 -> 64 3x3: 18 (38),
// 61x53x96x16 -> 32 5x5: 51 (452, element gather), 56x56x64x32 -> 128 3x3: 49
// (43); FP32 the last one: 123 (194), error against FP64 2.2e-7 (5.1e-7).
// Bound by the loads of whole channel rows from L2 (each tap group reads its
// pixels again) and, for FP32, by the six part products.
#include <algorithm>

#include "kcommon.hpp"
#include "nn_x3_parts.hpp"
#include "../nn_wgemm.hpp"

namespace afhip {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

enum WgMode : int { WG_BF16 = 0, WG_F16 = 1, WG_X3 = 2 };

struct WgParams {
    int N, H, W, C, K, OH, OW, fw, fh, RS;
    int s0, s1, p0, p1, d0, d1;
    int xpix, dpix;          // bytes of a pixel's channels in the copies
    int xs, ds;              // 32-channel slices
    int xbytes, dbytes;      // the copies (below 2^30)
    int npx, npd;            // pixels of x and dy
    int tilesK, tilesC, groups, ntile, nsplit;
    int slices, per;         // 32-pixel slices of dy, per split (a multiple of SL)
    int nbx, nbd;            // copy blocks (and flags) of x and dy
};

// Both channel-last copies in one launch, x first.
template <typename T>
__global__ __launch_bounds__(256) void wg_copies(T *__restrict__ xc, T *__restrict__ dc, const T *__restrict__ x,
                                                 const T *__restrict__ dy, WgParams p, unsigned *__restrict__ flags) {
    const bool first = (int)blockIdx.x < p.nbx;
    const int b = first ? (int)blockIdx.x : (int)blockIdx.x - p.nbx;
    const int hw = first ? p.H * p.W : p.OH * p.OW, Cd = first ? p.C : p.K, npix = first ? p.npx : p.npd;
    const int slices = first ? p.xs : p.ds;
    if constexpr (sizeof(T) == 4) {
        __shared__ unsigned tile[3][64 * 17];
        int flag = x3_copy_block(reinterpret_cast<uint16_t *>(first ? xc : dc), first ? x : dy, b, hw, Cd, npix,
                                 slices, tile);
        flag = x3_block_flags(flag);
        if (threadIdx.x == 0) flags[blockIdx.x] = (unsigned)flag;
    } else {
        // 64 pixels x 64 channels through LDS rows of 33 words
        __shared__ unsigned tile[64 * 33];
        const int ncg = (slices + 1) / 2, pb = b / ncg, c0 = (b - pb * ncg) * 64;
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int pix = min(pb * 64 + lane, npix - 1), n = pix / hw;
        const T *s = (first ? x : dy) + (long long)n * Cd * hw + (pix - n * hw);
        T v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = s[(long long)min(c0 + wave * 16 + u, Cd - 1) * hw];
        T *row = reinterpret_cast<T *>(tile + lane * 33) + wave * 16;
#pragma unroll
        for (int u = 0; u < 16; ++u) row[u] = c0 + wave * 16 + u < Cd ? v[u] : T{};
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = (int)threadIdx.x + 256 * u, px = e >> 3, g = e & 7;
            if (pb * 64 + px < npix && c0 + g * 8 < slices * 32) {
                const unsigned *q = tile + px * 33 + g * 4;
                *reinterpret_cast<uint4 *>((first ? xc : dc) + (long long)(pb * 64 + px) * (slices * 32) + c0 + g * 8) =
                    make_uint4(q[0], q[1], q[2], q[3]);
            }
        }
    }
}

// SL 32-pixel slices per stage, TT taps per workgroup.
template <int MODE, int SL, int TT>
__global__ __launch_bounds__(256, 2) void nn_wgemm_k(float *__restrict__ partial, const char *__restrict__ xc,
                                                     const char *__restrict__ dc, const unsigned *__restrict__ flags,
                                                     WgParams p) {
    constexpr int NP = MODE == WG_X3 ? 3 : 1;   // parts
    constexpr int PL = 4096 * SL;               // one part of one operand: 32 SL rows of 128 bytes
    __shared__ __attribute__((aligned(16))) char lds[(1 + TT) * NP * PL];

    // all tiles of a split on one XCD: they read the same pixels
    const int id = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int split = id / p.ntile;
    int tile = id - split * p.ntile;
    const int tg = tile / (p.tilesK * p.tilesC);
    tile -= tg * (p.tilesK * p.tilesC);
    const int k0 = tile / p.tilesC * 64, c0 = tile % p.tilesC * 64;
    const int t0 = tg * TT;
    const int sl0 = split * p.per, sl1 = min(sl0 + p.per, p.slices);
    const int q1 = min(sl1 * 32, p.npd);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = tid & 7, lrow = tid >> 3;
    const int ohw = p.OH * p.OW;

    int flag = 0;
    if constexpr (MODE == WG_X3) {
        // the flags of the blocks read: the split's pixels of dy, and of x the
        // rows from its first tap row to its last
        const int a = sl0 * 32, b = q1 - 1;
        const int na = a / ohw, nb = b / ohw, ya = (a - na * ohw) / p.OW, yb = (b - nb * ohw) / p.OW;
        const int lo = (na * p.H + min(max(ya * p.s1 - p.p1, 0), p.H - 1)) * p.W;
        const int hi = (nb * p.H + min(max(yb * p.s1 - p.p1 + (p.fh - 1) * p.d1, 0), p.H - 1)) * p.W + p.W - 1;
        const int fx1 = (hi / 64 + 1) * p.xs, fd1 = (b / 64 + 1) * p.ds;
        for (int f = lo / 64 * p.xs + tid; f < fx1; f += 256) flag |= (int)flags[f];
        for (int f = a / 64 * p.ds + tid; f < fd1; f += 256) flag |= (int)flags[p.nbx + f];
    }

    // the lane's 16 bytes of a pixel row
    const int xg = MODE == WG_X3 ? (c0 / 32 + (grp >> 2)) * 192 + (grp & 3) * 16 : c0 * 2 + grp * 16;
    const int dg = MODE == WG_X3 ? (k0 / 32 + (grp >> 2)) * 192 + (grp & 3) * 16 : k0 * 2 + grp * 16;
    const unsigned xout = c0 / 32 + (grp >> 2) < p.xs ? 0u : 0x80000000u;
    const unsigned dout = k0 / 32 + (grp >> 2) < p.ds ? 0u : 0x80000000u;
    int q[SL], n[SL], oh[SL], ow[SL];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        q[s] = (sl0 + s) * 32 + lrow;
        n[s] = q[s] / ohw;
        const int r = q[s] - n[s] * ohw;
        oh[s] = r / p.OW;
        ow[s] = r - oh[s] * p.OW;
    }
    // a stage on: 32 SL pixels
    const int en = 32 * SL / ohw, er = 32 * SL - en * ohw, eh = er / p.OW, ew = er - eh * p.OW;
    // taps past the last one repeat it and are not stored
    int ti[TT], tj[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int tc = min(t0 + t, p.RS - 1);
        tj[t] = tc / p.fw;
        ti[t] = tc - tj[t] * p.fw;
    }
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(xc), (short)0, p.xbytes, 0x00020000);
    const auto rd = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(dc), (short)0, p.dbytes, 0x00020000);
    uint4 sa[SL][NP], sb[SL][TT][NP];
    auto load = [&] {
#pragma unroll
        for (int s = 0; s < SL; ++s) {
            // outside the split or the image: past the end of the resource, as
            // an opaque mask (a condition would branch around the loads)
            unsigned past = q[s] < q1 ? 0u : 0x80000000u;
            asm volatile("" : "+v"(past));
            const unsigned doff = ((unsigned)q[s] * (unsigned)p.dpix + dg) | past | dout;
            const int iy = oh[s] * p.s1 - p.p1, ix = ow[s] * p.s0 - p.p0;
            const unsigned xoff = (unsigned)((n[s] * p.H + iy) * p.W + ix) * (unsigned)p.xpix + xg;
#pragma unroll
            for (int h = 0; h < NP; ++h)
                sa[s][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rd, (int)(doff + 64 * h), 0, 0));
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const int dyy = tj[t] * p.d1, dxx = ti[t] * p.d0;
                const bool in = (unsigned)(iy + dyy) < (unsigned)p.H && (unsigned)(ix + dxx) < (unsigned)p.W;
                unsigned off = xoff + (unsigned)((dyy * p.W + dxx) * p.xpix);
                off = (in ? off : 0x80000000u) | past | xout;
#pragma unroll
                for (int h = 0; h < NP; ++h)
                    sb[s][t][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(off + 64 * h), 0, 0));
            }
            q[s] += 32 * SL;
            ow[s] += ew;
            oh[s] += eh;
            n[s] += en;
            if (ow[s] >= p.OW) {
                ow[s] -= p.OW;
                ++oh[s];
            }
            if (oh[s] >= p.OH) {
                oh[s] -= p.OH;
                ++n[s];
            }
        }
    };
    // rows of 128 bytes, their four 32-byte blocks XORed by the row's eighth:
    // the 16 rows of a transposing read then fall into all banks twice
    char *slot = lds + lrow * 128 + (((grp >> 1) ^ (lrow >> 3 & 3)) * 32) + (grp & 1) * 16;
    const int wk = wave >> 1, wc = wave & 1, r16 = lane & 15, g4 = lane >> 4;
    const char *fr = lds + (8 * g4 + (r16 >> 2)) * 128 + (r16 & 3) * 8;
    auto frag = [&](int plane, int blk) {  // eight pixels of channel 16 blk + r16
        const char *b = fr + plane + ((blk ^ g4) * 32);
        const s16x4_t u = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)b);
        const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)(b + 512));
        return s16x8_t{u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]};
    };
    auto mma = [](s16x8_t a, s16x8_t b, f32x4_t c) {
        if constexpr (MODE == WG_F16)
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    };
    constexpr int LO = MODE == WG_X3 ? TT : 1;
    f32x4_t acc[TT][2][2], low[LO][2][2];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[t][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if constexpr (MODE == WG_X3) low[t][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }

    // a stage: pixels to LDS, the next stage's loads, mul per slice
    auto walk = [&](auto mul) {
        for (int k = sl0; k < sl1; k += SL) {
            __syncthreads();
#pragma unroll
            for (int s = 0; s < SL; ++s)
#pragma unroll
                for (int h = 0; h < NP; ++h) {
                    *reinterpret_cast<uint4 *>(slot + h * PL + s * 4096) = sa[s][h];
#pragma unroll
                    for (int t = 0; t < TT; ++t)
                        *reinterpret_cast<uint4 *>(slot + (NP + t * NP + h) * PL + s * 4096) = sb[s][t][h];
                }
            load();
            __syncthreads();
#pragma unroll
            for (int s = 0; s < SL; ++s) mul(s);
        }
    };
    load();
    if constexpr (MODE == WG_X3) flag = x3_block_flags(flag);
    if (MODE != WG_X3 || !(flag & X3_HUGE)) {
        walk([&](int s) {
            s16x8_t a[2][NP];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int h = 0; h < NP; ++h) a[i][h] = frag(h * PL + s * 4096, wk * 2 + i);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                s16x8_t b[2][NP];
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int h = 0; h < NP; ++h) b[j][h] = frag((NP + t * NP + h) * PL + s * 4096, wc * 2 + j);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[t][i][j] = mma(a[i][0], b[j][0], acc[t][i][j]);
                if constexpr (MODE == WG_X3) {
                    constexpr int PA[5] = {2, 0, 1, 1, 0}, PB[5] = {0, 2, 1, 0, 1};
#pragma unroll
                    for (int e = 0; e < 5; ++e)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j) low[t][i][j] = mma(a[i][PA[e]], b[j][PB[e]], low[t][i][j]);
                }
            }
        });
        if constexpr (MODE == WG_X3) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[t][i][j] = (acc[t][i][j] + low[t][i][j]) * X3_UNSCALE;
        }
    } else if constexpr (MODE == WG_X3) {
        walk([&](int s) {
            auto eight = [&](int plane, int blk, float (&v)[8]) {
                const s16x8_t a = frag(plane + s * 4096, blk), b = frag(plane + PL + s * 4096, blk),
                              c = frag(plane + 2 * PL + s * 4096, blk);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = x3_value((uint16_t)a[e], (uint16_t)b[e], (uint16_t)c[e]);
            };
            float a[2][8];
#pragma unroll
            for (int i = 0; i < 2; ++i) eight(0, wk * 2 + i, a[i]);
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float b[8];
                    eight((NP + t * NP) * PL, wc * 2 + j, b);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            acc[t][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[e], acc[t][i][j], 0, 0, 0);
                }
        });
    }

    // acc[t][i][j][v]: filter k0 + wk*32 + i*16 + 4*g4 + v, channel c0 + wc*32 + j*16 + r16
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        if (t0 + t >= p.RS) break;
        float *o = partial + ((long long)split * p.RS + t0 + t) * p.K * p.C;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int c = c0 + wc * 32 + j * 16 + r16;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int k = k0 + wk * 32 + i * 16 + 4 * g4 + v;
                    if (k < p.K && c < p.C) o[(long long)k * p.C + c] = acc[t][i][j][v];
                }
            }
    }
}

// dw[k][c][RS - 1 - t] = the splits' partials in order: a workgroup sums 64
// values, each wave a quarter of the splits (eight loads in flight), then the
// quarters.
template <typename TOut>
__global__ __launch_bounds__(256) void nn_wgemm_sum(TOut *__restrict__ dw, const float *__restrict__ partial,
                                                    WgParams p) {
    __shared__ float part[4][64];
    const int kc = p.K * p.C, total = p.RS * kc;  // below 2^29
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
    const int per = (p.nsplit + 3) / 4, s0 = w * per, s1 = min(s0 + per, p.nsplit);
    const float *src = partial + min(e, total - 1);
    float s = 0.f;
    int sp = s0;
    for (; sp + 8 <= s1; sp += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = src[(long long)(sp + k) * total];
#pragma unroll
        for (int k = 0; k < 8; ++k) s += v[k];
    }
    for (; sp < s1; ++sp) s += src[(long long)sp * total];
    part[w][threadIdx.x & 63] = s;
    __syncthreads();
    if (w || e >= total) return;
    s = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
    const int t = e / kc, r = e - t * kc;
    TOut *o = dw + (long long)r * p.RS + (p.RS - 1 - t);
    if constexpr (sizeof(TOut) == 4) *o = s;
    else if constexpr (__is_same(TOut, uint16_t)) *o = f32_to_bf16_bits(s);
    else *o = (_Float16)s;
}

// ---------------------------------------------------------------- host side
struct WgLayout {
    long long off_d = 0, off_flag = 0, off_part = 0, total = 0;
};
static bool wg_setup(int type, const long long *xd, const long long *wd, const long long *yd, const long long *st,
                     const long long *pd, const long long *dl, int cus, WgParams *p, WgLayout *L, int *tt) {
    const bool x3 = type == DT_F32;
    if (!x3 && type != DT_BF16 && type != DT_F16) return false;
    if (wd[2] != xd[2] || yd[2] != wd[3] || yd[3] != xd[3] || cus < 1) return false;
    for (int i = 0; i < 2; ++i)
        if (st[i] < 1 || dl[i] < 1) return false;
    const long long npx = xd[0] * xd[1] * xd[3], npd = yd[0] * yd[1] * yd[3], lim = 1LL << 30;  // offsets past a resource's end must not wrap
    if (npx < 1 || npd < 1 || wd[0] * wd[1] * wd[2] * wd[3] < 1) return false;
    const long long xs = (xd[2] + 31) / 32, ds = (wd[3] + 31) / 32, eb = x3 ? 192 : 64;
    if (npx * xs * eb >= lim || npd * ds * eb >= lim || wd[0] * wd[1] * wd[2] * wd[3] >= lim / 2) return false;
    p->W = (int)xd[0];
    p->H = (int)xd[1];
    p->C = (int)xd[2];
    p->N = (int)xd[3];
    p->fw = (int)wd[0];
    p->fh = (int)wd[1];
    p->K = (int)wd[3];
    p->OW = (int)yd[0];
    p->OH = (int)yd[1];
    p->s0 = (int)st[0];
    p->s1 = (int)st[1];
    p->p0 = (int)pd[0];
    p->p1 = (int)pd[1];
    p->d0 = (int)dl[0];
    p->d1 = (int)dl[1];
    p->RS = p->fw * p->fh;
    p->xs = (int)xs;
    p->ds = (int)ds;
    p->xpix = (int)(xs * eb);
    p->dpix = (int)(ds * eb);
    p->npx = (int)npx;
    p->npd = (int)npd;
    p->xbytes = (int)(npx * p->xpix);
    p->dbytes = (int)(npd * p->dpix);
    p->nbx = (int)((npx + 63) / 64 * (x3 ? xs : (xs + 1) / 2));
    p->nbd = (int)((npd + 63) / 64 * (x3 ? ds : (ds + 1) / 2));
    // three taps share the dy fragments where at most a tenth is wasted, one
    // tap at a time elsewhere. Three and one, us: 14x14x512x32 -> 512, 1x1, BF16
    // 32 and 24, FP32 77 and 48; 28x28x128x32 -> 128, 2x2, BF16 28.7 and 26.0,
    // FP32 55 and 50; 57x57x64x16 -> 64, 4x4, BF16 33.9 and 33.5, FP32 69 and 75.
    *tt = (p->RS + 2) / 3 * 30 <= 11 * p->RS ? 3 : 1;
    const int SL = x3 ? 1 : 2;
    p->tilesK = (p->K + 63) / 64;
    p->tilesC = (p->C + 63) / 64;
    p->groups = (p->RS + *tt - 1) / *tt;
    const long long ntile = (long long)p->tilesK * p->tilesC * p->groups;
    if (ntile >= (1LL << 24)) return false;
    p->ntile = (int)ntile;
    p->slices = (int)((npd + 31) / 32);
    // As many splits as two workgroups per CU hold, and not one more:
    // 28x28x128x64 -> 128, 3x3, FP32: 42 splits (504 of 512) 113 us, 43 (516) 157.
    // The 16-bit kernels, of which four fit, take twice as many where each has
    // pixels enough (32x32x96x64 -> 96, 5x5: 97 us against 110; 28x28x128x64 ->
    // 128, with 37 slices each of the larger share: 50 against 49) and half as many
    // where there are few, for the fewer partials to write and sum (17x80x64x16 ->
    // 128, 3x3: 23 us against 26; 21x70x3x34 -> 32, with 18 slices for each CU:
    // 24 against 23).
    const long long work = p->slices * ntile;
    const long long wide = x3 ? 2 : work > 112LL * cus ? 4 : work < 18LL * cus ? 1 : 2;
    long long split = std::max<long long>(1, wide * cus / ntile);
    const long long each = (long long)p->RS * p->K * p->C * 4;
    split = std::min<long long>(split, (p->slices + 4 * SL - 1) / (4 * SL));  // at least four stages each
    // few stages each: a workgroup per CU rather than two on a few of them
    // (28x28x128x16 -> 128, 3x3, stride 2, FP32: 252 workgroups 26 us, 300 33)
    if (x3 && split * ntile > cus && 2 * split * ntile < 3LL * cus) split = std::max<long long>(1, cus / ntile);
    split = std::max<long long>(1, std::min<long long>(split, (256LL << 20) / each));
    long long per = (p->slices + split - 1) / split;
    per = (per + SL - 1) / SL * SL;
    p->per = (int)per;
    p->nsplit = (int)((p->slices + per - 1) / per);
    auto al = [](long long b) { return (b + 255) & ~255LL; };
    L->off_d = al(p->xbytes);
    L->off_flag = L->off_d + al(p->dbytes);
    L->off_part = L->off_flag + (x3 ? al(4LL * (p->nbx + p->nbd)) : 0);
    L->total = L->off_part + each * p->nsplit;
    return true;
}

long long nn_wgemm_workspace(int type, const long long *xd, const long long *wd, const long long *yd,
                             const long long *st, const long long *pd, const long long *dl, int cus) {
    WgParams p;
    WgLayout L;
    int tt;
    return wg_setup(type, xd, wd, yd, st, pd, dl, cus, &p, &L, &tt) ? L.total : 0;
}

int nn_wgemm(int type, int out_type, void *dw, const void *x, const void *dy, const long long *xd, const long long *wd,
             const long long *yd, const long long *st, const long long *pd, const long long *dl, int cus, void *ws,
             long long ws_bytes, hipStream_t s) {
    WgParams p;
    WgLayout L;
    int tt;
    if (!wg_setup(type, xd, wd, yd, st, pd, dl, cus, &p, &L, &tt)) return K_ERR_NOT_SUPPORTED;
    if (out_type != DT_F32 && out_type != type) return K_ERR_TYPE;
    if (ws == nullptr || ws_bytes < L.total) return K_ERR_ARG;
    char *xc = (char *)ws, *dc = xc + L.off_d;
    unsigned *flags = (unsigned *)(xc + L.off_flag);
    float *part = (float *)(xc + L.off_part);
    const unsigned nb = (unsigned)(p.nbx + p.nbd), grid = (unsigned)p.ntile * p.nsplit;
    if (type == DT_F32)
        wg_copies<float><<<nb, 256, 0, s>>>((float *)xc, (float *)dc, (const float *)x, (const float *)dy, p, flags);
    else
        wg_copies<uint16_t><<<nb, 256, 0, s>>>((uint16_t *)xc, (uint16_t *)dc, (const uint16_t *)x,
                                               (const uint16_t *)dy, p, nullptr);
    auto fn = type == DT_F32    ? (tt == 3 ? nn_wgemm_k<WG_X3, 1, 3> : nn_wgemm_k<WG_X3, 1, 1>)
              : type == DT_BF16 ? (tt == 3 ? nn_wgemm_k<WG_BF16, 2, 3> : nn_wgemm_k<WG_BF16, 2, 1>)
                                : (tt == 3 ? nn_wgemm_k<WG_F16, 2, 3> : nn_wgemm_k<WG_F16, 2, 1>);
    fn<<<grid, 256, 0, s>>>(part, xc, dc, flags, p);
    const unsigned sb = (unsigned)(((long long)p.RS * p.K * p.C + 63) / 64);
    if (out_type == DT_F32)
        nn_wgemm_sum<float><<<sb, 256, 0, s>>>((float *)dw, part, p);
    else if (out_type == DT_BF16)
        nn_wgemm_sum<uint16_t><<<sb, 256, 0, s>>>((uint16_t *)dw, part, p);
    else
        nn_wgemm_sum<_Float16><<<sb, 256, 0, s>>>((_Float16 *)dw, part, p);
    return launch_status();
}

}  // namespace afhip
