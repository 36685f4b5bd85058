// convolve2_nn forward, data gradient and filter gradient as implicit GEMMs
// on the gfx950 matrix cores.
//
// Reference semantics (src/backend/cpu/convolve.cpp:123-243; closed forms):
//   fwd   y[ow,oh,k,n]  = sum_{c,i,j} x[ow*s0-p0+i*d0, oh*s1-p1+j*d1, c, n]
//                                     * w[fw-1-i, fh-1-j, c, k]
//   dgrad dx[x,y,c,n]   = sum over (k,ow,oh,i,j) hitting (x,y) of dy*w(flipped)
//   wgrad dw[fw-1-i, fh-1-j, c, k] = sum_{n,ow,oh} x[...] * dy[ow,oh,k,n]
// ArrayFire dims [W,H,C,N] are row-major NCHW; [fw,fh,C,K] is KCRS.
//
// GEMM views (C[M x Ncol] += A[M x R] * B[R x Ncol]):
//   fwd   M = K,  Ncol = N*OH*OW, R = (tap, C)   A = w,  B = im2col(x)
//   dgrad M = C,  Ncol = N*H*W,   R = (tap, K)   A = w,  B = col(dy) gathered
//                                                through the stride phases
//   wgrad M = K,  Ncol = C*fh*fw, R = N*OH*OW    A = dy, B = im2col(x)^T.
// Layers with too few output tiles to fill the chip split R across
// workgroups (FP32 partial tiles, then a second pass that sums them in split
// order: deterministic). A strided data gradient orders its columns by stride
// phase (x mod s0, y mod s1), each phase padded to whole tiles, and visits
// only the taps that reach that phase: about 1/(s0*s1) of the slices.
// Nothing is materialised: each 32-deep slice of R is gathered from HBM into
// registers, converted to the operand format and stored to LDS with R
// contiguous per row, where the MFMA fragments read it with ds_read_b128.
//
// Workgroup: 256 lanes (4 waves as 2x2), output tile 128 x 128, each wave a
// 64 x 64 block of 4x4 MFMA 16x16 tiles. Operand formats (MODE):
//   F32   v_mfma_f32_16x16x4_f32, FP32 operands
//   BF16  v_mfma_f32_16x16x32_bf16, operands rounded to bf16 (RNE)
//   F16   v_mfma_f32_16x16x32_f16
//   SPLIT hi = bf16(v), lo = bf16(v - hi); hi*hi' + hi*lo' + lo*hi' on BF16
// Accumulation is FP32 in every mode. One LDS buffer; the next slice's global
// loads are in flight in registers while the current slice is multiplied.
// nn_gemm gathers its operands element by element and takes any geometry and
// conversion; nn_clgemm (below) reads channel-last copies where the operands
// are stored in the MMA type.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "kcommon.hpp"
#include "nn_x3_parts.hpp"
#include "../nn_x3.hpp"
#include "../../../include/afhip_kernels.h"

namespace afhip {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));

enum Mode : int { M_F32 = 0, M_BF16 = 1, M_F16 = 2, M_SPLIT = 3 };
enum Pass : int { P_FWD = 0, P_DGRAD = 1, P_WGRAD = 2 };

// Strided data gradients order their columns by stride phase when there are
// at most this many phases (s0 * s1).
constexpr int kMaxPhases = 256;

struct NNParams {
    // x [W,H,C,N], w [fw,fh,C,K], y [OW,OH,K,N]
    int W, H, C, N, fw, fh, K, OW, OH;
    int s0, s1, p0, p1, d0, d1;
    int RS;              // fw*fh
    long long M, Ncol;   // GEMM extents
    int R;               // reduction extent (wgrad) -- informational
    int kchunks;         // 32-deep slices per tap (fwd: ceil(C/32), dgrad: ceil(K/32))
    long long ksteps;    // total slices (phased data gradient: the most of any phase)
    long long ksteps_per_split;
    int nsplit;          // > 1: FP32 partial tiles per split, summed by nn_split_reduce / wgrad_reduce
    long long tilesM, tilesN;
    // Phased data gradient (stride > 1): the input pixels (x, y) with
    // x = s0*mx + rx, y = s1*my + ry form phase ph = ry*s0 + rx; each phase's
    // N*My*Mx columns start at column tile ph_tile0[ph] and only the taps
    // (i, j) with (rx + p0 - i*d0) and (ry + p1 - j*d1) divisible by the
    // strides meet them, so only those taps are visited.
    int phased;
    int nph;
    int ph_tile0[kMaxPhases + 1];
    // Channel-last operands (forward and data gradient, operands stored in
    // the MMA type): packed weights Wp [RS][M][Rcp] and the activation (x,
    // or dy for the data gradient) as [N][rows][cols][Rcp], Rcp = the
    // reduction channels rounded up to the 32-deep slice, zero past them.
    int cl;
    int Rcp;
    int wp_bytes, act_bytes;  // sizes of the channel-last copies (each below 2^31 - 64)
    int nsplit_req;           // > 0: the caller's split count (forward / data gradient)
};

// Phase extents: pixels of residue r along an axis of length L and stride s,
// and the taps of a filter (length f, dilation d, padding pd) that reach them.
__host__ __device__ inline int phase_len(int L, int s, int r) { return r < L ? (L - r + s - 1) / s : 0; }
__host__ __device__ inline bool phase_tap(int r, int pd, int i, int d, int s) {
    const int v = (r + pd - i * d) % s;
    return v == 0;
}
__host__ __device__ inline int phase_taps(int f, int r, int pd, int d, int s) {
    int n = 0;
    for (int i = 0; i < f; ++i) n += phase_tap(r, pd, i, d, s) ? 1 : 0;
    return n;
}
// The u-th tap (in increasing order) that reaches residue r.
__host__ __device__ inline int phase_tap_at(int f, int r, int pd, int d, int s, int u) {
    for (int i = 0; i < f; ++i)
        if (phase_tap(r, pd, i, d, s)) {
            if (u == 0) return i;
            --u;
        }
    return 0;
}

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int NT = 256;

// ------------------------------------------------------------- element IO
struct bf16s {
    uint16_t b;
};
template <typename T>
__device__ inline float ld_f(const T *p, long long i);
template <>
__device__ inline float ld_f<float>(const float *p, long long i) {
    return p[i];
}
template <>
__device__ inline float ld_f<bf16s>(const bf16s *p, long long i) {
    return bf16_bits_to_f32(p[i].b);
}
template <>
__device__ inline float ld_f<_Float16>(const _Float16 *p, long long i) {
    return (float)p[i];
}

template <typename T>
__device__ inline void st_f(T *p, long long i, float v);
template <>
__device__ inline void st_f<float>(float *p, long long i, float v) {
    p[i] = v;
}
template <>
__device__ inline void st_f<bf16s>(bf16s *p, long long i, float v) {
    p[i].b = f32_to_bf16_bits(v);
}
template <>
__device__ inline void st_f<_Float16>(_Float16 *p, long long i, float v) {
    p[i] = (_Float16)v;
}

__device__ inline uint16_t f32_to_f16_bits(float v) {
    _Float16 h = (_Float16)v;
    return __builtin_bit_cast(uint16_t, h);
}

// ------------------------------------------------------------- LDS layout
// Each operand tile is 128 rows x 32 R-values. 16-bit formats use a row pitch
// of 40 elements (80 B), FP32 a pitch of 36 (144 B); the pad staggers rows
// across LDS banks for the 16-byte fragment reads.
template <int MODE>
struct Lds {
    static constexpr int PITCH = MODE == M_F32 ? 36 : 40;
    static constexpr int ESZ = MODE == M_F32 ? 4 : 2;
    static constexpr int PARTS = MODE == M_SPLIT ? 2 : 1;  // hi, lo
    static constexpr int TILE_BYTES = 128 * PITCH * ESZ;
    static constexpr int BYTES = 2 * PARTS * TILE_BYTES;    // A and B
};

// Writes 16 values (one row, R offset kk0) of an operand tile.
template <int MODE>
__device__ inline void store_row16(char *tile, int row, int kk0, const float (&v)[16]) {
    constexpr int P = Lds<MODE>::PITCH;
    if constexpr (MODE == M_F32) {
        float *t = reinterpret_cast<float *>(tile) + row * P + kk0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4 *>(t + 4 * q) =
                make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    } else if constexpr (MODE == M_BF16 || MODE == M_F16) {
        uint16_t *t = reinterpret_cast<uint16_t *>(tile) + row * P + kk0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            u16x8_t h;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                h[e] = MODE == M_BF16 ? f32_to_bf16_bits(v[8 * q + e]) : f32_to_f16_bits(v[8 * q + e]);
            *reinterpret_cast<u16x8_t *>(t + 8 * q) = h;
        }
    } else {  // SPLIT: hi tile then lo tile
        uint16_t *th = reinterpret_cast<uint16_t *>(tile) + row * P + kk0;
        uint16_t *tl = reinterpret_cast<uint16_t *>(tile + Lds<MODE>::TILE_BYTES) + row * P + kk0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            u16x8_t hh, ll;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = v[8 * q + e];
                const uint16_t hb = f32_to_bf16_bits(x);
                hh[e] = hb;
                ll[e] = f32_to_bf16_bits(x - bf16_bits_to_f32(hb));
            }
            *reinterpret_cast<u16x8_t *>(th + 8 * q) = hh;
            *reinterpret_cast<u16x8_t *>(tl + 8 * q) = ll;
        }
    }
}

// One 32-deep slice: acc[4][4] += A(wave rows) * B(wave cols).
template <int MODE>
__device__ inline void mma_slice(const char *tA, const char *tB, int wm, int wn, int lane,
                                 f32x4_t (&acc)[4][4]) {
    constexpr int P = Lds<MODE>::PITCH;
    const int r16 = lane & 15, g = lane >> 4;
    if constexpr (MODE == M_F32) {
        const float *a = reinterpret_cast<const float *>(tA);
        const float *b = reinterpret_cast<const float *>(tB);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4 af[4], bfr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                af[i] = *reinterpret_cast<const float4 *>(a + (wm * 64 + i * 16 + r16) * P + h * 16 + 4 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bfr[j] = *reinterpret_cast<const float4 *>(b + (wn * 64 + j * 16 + r16) * P + h * 16 + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].x, bfr[j].x, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].y, bfr[j].y, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].z, bfr[j].z, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].w, bfr[j].w, acc[i][j], 0, 0, 0);
                }
        }
    } else {
        const uint16_t *a = reinterpret_cast<const uint16_t *>(tA);
        const uint16_t *b = reinterpret_cast<const uint16_t *>(tB);
        u16x8_t af[4], bfr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            af[i] = *reinterpret_cast<const u16x8_t *>(a + (wm * 64 + i * 16 + r16) * P + 8 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            bfr[j] = *reinterpret_cast<const u16x8_t *>(b + (wn * 64 + j * 16 + r16) * P + 8 * g);
        if constexpr (MODE == M_SPLIT) {
            constexpr int TB = Lds<MODE>::TILE_BYTES / 2;  // elements per tile
            u16x8_t al[4], bl[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                al[i] = *reinterpret_cast<const u16x8_t *>(a + TB + (wm * 64 + i * 16 + r16) * P + 8 * g);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bl[j] = *reinterpret_cast<const u16x8_t *>(b + TB + (wn * 64 + j * 16 + r16) * P + 8 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bf16x8_t ah = __builtin_bit_cast(bf16x8_t, af[i]);
                    const bf16x8_t bh = __builtin_bit_cast(bf16x8_t, bfr[j]);
                    const bf16x8_t alo = __builtin_bit_cast(bf16x8_t, al[i]);
                    const bf16x8_t blo = __builtin_bit_cast(bf16x8_t, bl[j]);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alo, bh, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, blo, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc[i][j], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if constexpr (MODE == M_BF16) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, af[i]), __builtin_bit_cast(bf16x8_t, bfr[j]),
                            acc[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(f16x8_t, af[i]), __builtin_bit_cast(f16x8_t, bfr[j]),
                            acc[i][j], 0, 0, 0);
                    }
                }
        }
    }
}

// ------------------------------------------------------------- gathers
// Each lane owns one row of the A tile and one row of the B tile and fills
// 16 consecutive R positions of each (kk0 = 0 or 16).

// fwd / wgrad helper: output pixel q -> (n, oh, ow)
struct Pix {
    int n, a, b;  // image, row, column
};
__device__ inline Pix decode(long long q, int rows, int cols) {
    Pix p;
    const long long per = (long long)rows * cols;
    p.n = (int)(q / per);
    const int r = (int)(q - (long long)p.n * per);
    p.a = r / cols;
    p.b = r - p.a * cols;
    return p;
}

template <typename TIn, int PASS>
struct Gather;

// ---- forward: A = w (row k), B = im2col(x) (row = output pixel)
template <typename TIn>
struct Gather<TIn, P_FWD> {
    const TIn *x, *w;
    const NNParams &p;
    long long arow, brow;  // global row indices
    bool bvalid;
    Pix bp;
    __device__ Gather(const TIn *x_, const TIn *w_, const NNParams &p_, long long ar, long long br, int)
        : x(x_), w(w_), p(p_), arow(ar), brow(br) {
        bvalid = br < p.Ncol;
        bp = decode(bvalid ? br : 0, p.OH, p.OW);
    }
    // slice -> (tap, channel block)
    __device__ void load(long long ks, int kk0, float (&va)[16], float (&vb)[16]) const {
        const int t = (int)(ks / p.kchunks);
        const int c0 = (int)(ks - (long long)t * p.kchunks) * BK + kk0;
        const int i = t % p.fw, j = t / p.fw;
        // A: w[k][c][fh-1-j][fw-1-i]
        const bool ak = arow < p.K;
        const long long abase = (arow * p.C) * p.RS + (p.RS - 1 - t);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int c = c0 + e;
            va[e] = (ak && c < p.C) ? ld_f(w, abase + (long long)c * p.RS) : 0.f;
        }
        // B: x[n][c][oh*s1-p1+j*d1][ow*s0-p0+i*d0]
        const int ih = bp.a * p.s1 - p.p1 + j * p.d1;
        const int iw = bp.b * p.s0 - p.p0 + i * p.d0;
        const bool ok = bvalid && ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
        const long long hw = (long long)p.H * p.W;
        const long long bbase = ((long long)bp.n * p.C) * hw + (long long)ih * p.W + iw;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int c = c0 + e;
            vb[e] = (ok && c < p.C) ? ld_f(x, bbase + (long long)c * hw) : 0.f;
        }
    }
};

// ---- data gradient: A = w (row c), B = dy gathered (row = input pixel)
template <typename TIn>
struct Gather<TIn, P_DGRAD> {
    const TIn *dy, *w;
    const NNParams &p;
    long long arow;
    bool bvalid;
    int bn, by, bx;     // this lane's B row: image and input pixel
    int rx, ry, Ti;     // phased: the tile's phase and its tap count along W
    __device__ Gather(const TIn *dy_, const TIn *w_, const NNParams &p_, long long ar, long long br, int ph)
        : dy(dy_), w(w_), p(p_), arow(ar) {
        if (p.phased) {
            rx = ph % p.s0;
            ry = ph / p.s0;
            const int Mx = phase_len(p.W, p.s0, rx), My = phase_len(p.H, p.s1, ry);
            bvalid = br < (long long)p.N * My * Mx;
            const Pix q = decode(bvalid ? br : 0, My, Mx);
            bn = q.n;
            by = p.s1 * q.a + ry;
            bx = p.s0 * q.b + rx;
            Ti = phase_taps(p.fw, rx, p.p0, p.d0, p.s0);
        } else {
            rx = ry = 0;
            Ti = p.fw;
            bvalid = br < p.Ncol;
            const Pix q = decode(bvalid ? br : 0, p.H, p.W);
            bn = q.n;
            by = q.a;
            bx = q.b;
        }
    }
    __device__ void load(long long ks, int kk0, float (&va)[16], float (&vb)[16]) const {
        const int u = (int)(ks / p.kchunks);
        const int k0 = (int)(ks - (long long)u * p.kchunks) * BK + kk0;
        int i, j;
        if (p.phased) {
            const int ui = u % Ti;
            i = phase_tap_at(p.fw, rx, p.p0, p.d0, p.s0, ui);
            j = phase_tap_at(p.fh, ry, p.p1, p.d1, p.s1, u / Ti);
        } else {
            i = u % p.fw;
            j = u / p.fw;
        }
        const int t = j * p.fw + i;
        // A: w[k][c][fh-1-j][fw-1-i], row = c, R = k
        const bool ac = arow < p.C;
        const long long crs = (long long)p.C * p.RS;
        const long long abase = arow * p.RS + (p.RS - 1 - t);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int k = k0 + e;
            va[e] = (ac && k < p.K) ? ld_f(w, abase + (long long)k * crs) : 0.f;
        }
        // B: dy[n][k][oh][ow] where oh*s1 - p1 + j*d1 = y, ow*s0 - p0 + i*d0 = x
        const int nh = by + p.p1 - j * p.d1;
        const int nw = bx + p.p0 - i * p.d0;
        bool ok = bvalid && nh >= 0 && nw >= 0 && (nh % p.s1) == 0 && (nw % p.s0) == 0;
        const int oh = ok ? nh / p.s1 : 0, ow = ok ? nw / p.s0 : 0;
        ok = ok && oh < p.OH && ow < p.OW;
        const long long ohw = (long long)p.OH * p.OW;
        const long long bbase = ((long long)bn * p.K) * ohw + (long long)oh * p.OW + ow;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int k = k0 + e;
            vb[e] = (ok && k < p.K) ? ld_f(dy, bbase + (long long)k * ohw) : 0.f;
        }
    }
};

// ---- filter gradient: A = dy (row k, R = output pixel), B = x (row = (c,tap))
template <typename TIn>
struct Gather<TIn, P_WGRAD> {
    const TIn *x, *dy;
    const NNParams &p;
    long long arow, brow;
    int bc, bi, bj;  // B row -> channel and tap (i along W, j along H)
    bool bvalid;
    __device__ Gather(const TIn *x_, const TIn *dy_, const NNParams &p_, long long ar, long long br, int)
        : x(x_), dy(dy_), p(p_), arow(ar), brow(br) {
        bvalid = br < p.Ncol;
        const int r = bvalid ? (int)br : 0;
        bc = r / p.RS;
        const int t = r - bc * p.RS;
        bi = t % p.fw;
        bj = t / p.fw;
    }
    __device__ void load(long long ks, int kk0, float (&va)[16], float (&vb)[16]) const {
        const long long q0 = ks * BK + kk0;
        const long long Rtot = (long long)p.N * p.OH * p.OW;
        Pix pp = decode(q0 < Rtot ? q0 : 0, p.OH, p.OW);
        const long long ohw = (long long)p.OH * p.OW, hw = (long long)p.H * p.W;
        const bool ak = arow < p.K;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const bool inr = q0 + e < Rtot;
            // A: dy[n][k][oh][ow]
            va[e] = (ak && inr) ? ld_f(dy, ((long long)pp.n * p.K + arow) * ohw + (long long)pp.a * p.OW + pp.b)
                                : 0.f;
            // B: x[n][c][oh*s1-p1+j*d1][ow*s0-p0+i*d0]
            const int ih = pp.a * p.s1 - p.p1 + bj * p.d1;
            const int iw = pp.b * p.s0 - p.p0 + bi * p.d0;
            const bool ok = bvalid && inr && ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
            vb[e] = ok ? ld_f(x, ((long long)pp.n * p.C + bc) * hw + (long long)ih * p.W + iw) : 0.f;
            // next pixel
            if (++pp.b == p.OW) {
                pp.b = 0;
                if (++pp.a == p.OH) {
                    pp.a = 0;
                    ++pp.n;
                }
            }
        }
    }
};

// ------------------------------------------------- channel-last GEMM
// Operands stored in the MMA type run here. They are first copied channel-last: the weights
// as Wp [RS][M][Rcp] (forward M = K, R = C, Wp[t][k][c] =
// w[k][c][fh-1-j][fw-1-i]; data gradient M = C, R = K, Wp[t][c][k] = the same
// element; t = j*fw + i) and the activation as [N][rows][cols][Rcp], zeros
// past the reduction channels.

// Both copies in one launch. The first nbw workgroups pack the weights, one
// element per lane; each of the others transposes 64 pixels by 128 bytes of
// channels through LDS, so that a wave reads 64 consecutive pixels of a
// channel and writes whole 128-byte channel runs (an LDS row is 33 words: the
// 64 pixels of a wave's write fall into 64 banks).
template <typename T>
__global__ __launch_bounds__(256) void nn_cl_copies(T *__restrict__ wp, const T *__restrict__ w, NNParams p,
                                                    int dgrad, int nbw, T *__restrict__ dst,
                                                    const T *__restrict__ src, int hw, int Cd, int npix, int ncg) {
    if ((int)blockIdx.x < nbw) {
        const int Rc = dgrad ? p.K : p.C, M = (int)p.M;
        const unsigned total = (unsigned)(p.RS * M) * (unsigned)p.Rcp;  // below 2^31
        for (unsigned e = blockIdx.x * 256u + threadIdx.x; e < total; e += (unsigned)nbw * 256u) {
            const unsigned mt = e / (unsigned)p.Rcp;
            const int r = (int)(e - mt * (unsigned)p.Rcp);
            const int t = (int)(mt / (unsigned)M), m = (int)mt - t * M;
            T v{};
            if (r < Rc) {
                const int k = dgrad ? r : m, c = dgrad ? m : r;
                v = w[((long long)k * p.C + c) * p.RS + (p.RS - 1 - t)];
            }
            wp[e] = v;
        }
        return;
    }
    constexpr int CH = 128 / (int)sizeof(T);
    __shared__ unsigned tile[64 * 33];
    const unsigned b = blockIdx.x - nbw;
    const int pb = (int)(b / (unsigned)ncg), c0 = (int)(b - (unsigned)pb * ncg) * CH;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int pix = pb * 64 + lane;
    const int n = min(pix, npix - 1) / hw;
    const T *s = src + (long long)n * Cd * hw + (min(pix, npix - 1) - n * hw);
    T v[CH / 4];
#pragma unroll
    for (int u = 0; u < CH / 4; ++u) {
        const int c = c0 + wave * (CH / 4) + u;
        v[u] = s[(long long)min(c, Cd - 1) * hw];
    }
    T *row = reinterpret_cast<T *>(tile + lane * 33) + wave * (CH / 4);
#pragma unroll
    for (int u = 0; u < CH / 4; ++u) row[u] = c0 + wave * (CH / 4) + u < Cd ? v[u] : T{};
    __syncthreads();
    // 64 pixels x 8 groups of 16 bytes
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = (int)threadIdx.x + 256 * u, px = e >> 3, g = e & 7;
        const int ch = c0 + g * (16 / (int)sizeof(T));
        if (pb * 64 + px < npix && ch < p.Rcp) {
            const unsigned *q = tile + px * 33 + g * 4;
            *reinterpret_cast<uint4 *>(dst + (long long)(pb * 64 + px) * p.Rcp + ch) = make_uint4(q[0], q[1], q[2], q[3]);
        }
    }
}

// The taps a tile visits, as shifts of its pixels in the activation: tap (i, j)
// of the walk reads column X + sx0 + i*dsx of row Y + sy0 + j*dsy and holds
// filter tap t = (j0 + j*js)*fw + i0 + i*is. Forward: every tap, X = ow*s0.
// Data gradient: the taps that reach the tile's stride phase, in the phase's
// own pixel grid (all of them at stride 1).
struct TapAxis {
    int n, start, step, i0, is;
};
__device__ inline TapAxis tap_axis(bool fwd, bool phased, int f, int pd, int d, int s, int r) {
    TapAxis a;
    if (fwd || !phased) {
        a.n = f;
        a.i0 = 0;
        a.is = 1;
        a.start = fwd ? -pd : pd;
        a.step = fwd ? d : -d;
        return a;
    }
    // residues i with (r + pd - i*d) divisible by s: an arithmetic progression
    a.n = a.i0 = 0;
    a.is = 1;
    int first = -1, second = -1;
    for (int i = 0; i < f; ++i)
        if (phase_tap(r, pd, i, d, s)) {
            if (first < 0) first = i;
            else if (second < 0) second = i;
            ++a.n;
        }
    if (a.n) a.i0 = first;
    if (a.n > 1) a.is = second - first;
    a.start = (r + pd - a.i0 * d) / s;
    a.step = -(a.is * d) / s;
    return a;
}

// A workgroup's tile: split, first channel and column, its stride phase and
// pixel grid.
struct ClTile {
    int split, m0, n0, ph, rx, ry, gw, gh, ncol;
    bool phased;
};
template <int PASS, int TM, int TN>
__device__ __forceinline__ ClTile cl_tile(const NNParams &p) {
    ClTile t;
    const unsigned tiles = (unsigned)(p.tilesM * p.tilesN), bid = blockIdx.x;
    t.split = (int)(bid / tiles);
    const unsigned tl = bid - t.split * tiles;
    const int tm = (int)(tl / (unsigned)p.tilesN), tn = (int)(tl - tm * (unsigned)p.tilesN);
    t.m0 = tm * TM;
    t.n0 = tn * TN;
    t.phased = PASS == P_DGRAD && p.phased;
    t.ph = t.rx = t.ry = 0;
    if (t.phased) {  // phases start on whole tiles of BN columns
        while (t.ph + 1 < p.nph && t.n0 >= p.ph_tile0[t.ph + 1] * BN) ++t.ph;
        t.n0 -= p.ph_tile0[t.ph] * BN;
        t.rx = t.ph % p.s0;
        t.ry = t.ph / p.s0;
        t.gw = phase_len(p.W, p.s0, t.rx);
        t.gh = phase_len(p.H, p.s1, t.ry);
    } else {
        t.gw = PASS == P_FWD ? p.OW : p.W;
        t.gh = PASS == P_FWD ? p.OH : p.H;
    }
    t.ncol = p.N * t.gw * t.gh;  // columns of the grid
    return t;
}

// Results of a wave's TM/2 x TN/2 block: to the split's partial tile, or to the
// output by way of LDS (lds: the staging buffer, free by now), so that a wave
// stores a channel's 64 neighbouring pixels at once, four of them per lane
// where planes are whole groups of four. Straight from the registers a store
// instruction touches 16 channels, 64 cache lines with single pixels: the
// 75x61x64x16 -> 128 stride 2 layer, BF16, forward 23.5 us with its copies and
// 21.3 by LDS, its data gradient 33.9 and 28.3; 56x56x64x32 -> 128 in FP32 by
// parts 119 and 116 us.
template <typename TOut, int PASS, int TM, int TN>
__device__ __forceinline__ void cl_store(TOut *__restrict__ out, float *__restrict__ partial,
                                         const f32x4_t (&acc)[TM / 32][TN / 32], const NNParams &p, const ClTile &t,
                                         int wm, int wn, int r16, int g4, char *lds) {
    constexpr int MI = TM / 32, NJ = TN / 32;
    const int m0 = t.m0, n0 = t.n0, ph = t.ph, rx = t.rx, ry = t.ry, gw = t.gw, gh = t.gh, ncol = t.ncol;
    const bool phased = t.phased;
    const int split = t.split;
    // acc[i][j][v]: channel m0 + wm*TM/2 + i*16 + r16, column n0 + wn*TN/2 + j*16 + 4*g4 + v
    const int mlane = m0 + wm * (TM / 2) + r16;
    if (p.nsplit > 1) {
        const int pc0 = phased ? p.ph_tile0[ph] * BN : 0, nall = (int)p.Ncol;
        float *pt = partial + (long long)split * p.M * p.Ncol;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int col = pc0 + n0 + wn * (TN / 2) + j * 16 + 4 * g4;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int m = mlane + 16 * i;
                if (m >= (int)p.M) continue;
                float *o = pt + (long long)m * nall + col;
                if ((nall & 3) == 0 && col + 4 <= nall) {
                    *reinterpret_cast<float4 *>(o) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (col + v < nall) o[v] = acc[i][j][v];
                }
            }
        }
        return;
    }
    const unsigned per = (unsigned)(gw * gh);
    const long long plane = PASS == P_FWD ? (long long)p.OH * p.OW : (long long)p.H * p.W;
    constexpr int E = (int)sizeof(TOut), PITCH = TN * E + 16;
    // 128 x 128 FP32 results go through LDS half a tile of channels at a time
    constexpr int PARTS = TM * PITCH > 2 * (TM + TN) * 128 ? 2 : 1, MP = TM / PARTS;
    const bool vec = !phased && (plane & 3) == 0 && ((uintptr_t)out & (4 * sizeof(TOut) - 1)) == 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int part = 0; part < PARTS; ++part) {
        __syncthreads();
        if (PARTS == 1 || wm == part) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    TOut r[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v) st_f(r, v, acc[i][j][v]);
                    char *o = lds + ((PARTS == 1 ? wm * (TM / 2) : 0) + i * 16 + r16) * PITCH +
                              (wn * (TN / 2) + j * 16 + 4 * g4) * E;
                    if constexpr (E == 4)
                        *reinterpret_cast<uint4 *>(o) = __builtin_bit_cast(uint4, r);
                    else
                        *reinterpret_cast<uint2 *>(o) = __builtin_bit_cast(uint2, r);
                }
        }
        __syncthreads();
        const int mbase = m0 + part * MP;
        if (vec) {
            // lane: four pixels of row lane / (TN / 4)
            constexpr int LPR = TN / 4, RPW = 64 / LPR;
            const int px = (lane % LPR) * 4, col = n0 + px;
            if (col < ncol) {
                const unsigned n = (unsigned)col / per;
                TOut *o = out + (long long)n * p.M * plane + (col - n * per);
#pragma unroll 4
                for (int m = wave * RPW + lane / LPR; m < MP; m += 4 * RPW) {
                    if (mbase + m >= (int)p.M) break;
                    const char *q = lds + m * PITCH + px * E;
                    if constexpr (E == 4)
                        *reinterpret_cast<uint4 *>(o + (mbase + m) * plane) = *reinterpret_cast<const uint4 *>(q);
                    else
                        *reinterpret_cast<uint2 *>(o + (mbase + m) * plane) = *reinterpret_cast<const uint2 *>(q);
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < TN / 64; ++h) {
                const int px = lane + 64 * h, col = n0 + px;
                if (col >= ncol) continue;
                const unsigned n = (unsigned)col / per, yx = col - n * per;
                long long at = (long long)n * p.M * plane;
                if (phased) {
                    const int y = (int)(yx / (unsigned)gw), x = (int)yx - y * gw;
                    at += (long long)(p.s1 * y + ry) * p.W + p.s0 * x + rx;
                } else {
                    at += yx;
                }
#pragma unroll 4
                for (int m = wave; m < MP; m += 4) {
                    if (mbase + m >= (int)p.M) break;
                    out[at + (mbase + m) * plane] = *reinterpret_cast<const TOut *>(lds + m * PITCH + px * E);
                }
            }
        }
    }
}

// Output tile TM x TN per 256-lane workgroup, 2 x 2 waves. R is walked in
// stages of 128 bytes per row: two 32-deep slices of 16-bit operands, one of
// FP32, in the slice order of nn_gemm, so both give the same bits. LDS rows
// are 128 bytes with their eight 16-byte groups XORed by the row, which keeps
// the fragments' 16-byte reads free of bank conflicts without padding.
// DEPTH register sets and two LDS buffers: a stage's loads are issued DEPTH
// stages ahead and stored one stage ahead, with one barrier per stage. Every
// lane follows the walk over (tap, channel slice) with counters of its own;
// pixels outside the activation read zeros past the end of the buffer resource.
// What bounds small layers is the latency of each stage's loads (the copies
// were just written by other XCDs and come from the Infinity Cache, about a
// microsecond away), which the depth covers, and the walk's address arithmetic
// (about 50 instructions per stage beside 8 to 32 MFMAs). Copies included:
// 27x27x96x16 -> 128, 5x5, F16 29 us (40 us before, of which 9 to sum splits);
// 28x28x128x16 -> 128, 3x3, stride 2, BF16 15 us (25); its data gradient 17 us
// (38); 75x70x128x8 -> 256, 3x3, BF16 58 us, 425 TFLOP/s (90 us on conv_patch).
// Two stages of 256 bytes per row in place of four of 128 were no faster on
// small layers (33 us for the 5x5) and slower on large ones (84 us).
template <int MODE, typename T, typename TOut, int PASS, int TM, int TN>
__global__ __launch_bounds__(NT, 2) void nn_clgemm(TOut *__restrict__ out, const T *__restrict__ act,
                                                   const T *__restrict__ wp, float *__restrict__ partial,
                                                   NNParams p) {
    constexpr int SB = 128, DEPTH = TM + TN > 192 ? 2 : 4;
    constexpr int E = (int)sizeof(T), CPS = SB / (32 * E);  // 32-deep slices per stage
    constexpr int G = SB / 16, GPC = G / CPS;               // 16-byte groups per row, per slice
    constexpr int RP = NT / G;                              // rows per load of the workgroup
    constexpr int NA = TM / RP, NB = TN / RP;               // loads per lane and stage
    constexpr int MI = TM / 32, NJ = TN / 32;               // 16 x 16 results per wave
    __shared__ __attribute__((aligned(16))) char lds[2][(TM + TN) * SB];

    const ClTile t0 = cl_tile<PASS, TM, TN>(p);
    const int split = t0.split, m0 = t0.m0, n0 = t0.n0, rx = t0.rx, ry = t0.ry, gw = t0.gw, gh = t0.gh, ncol = t0.ncol;
    const bool phased = t0.phased;
    if (n0 >= ncol) return;  // a phase's padding
    const TapAxis ax = tap_axis(PASS == P_FWD, phased, p.fw, p.p0, p.d0, p.s0, rx);
    const TapAxis ay = tap_axis(PASS == P_FWD, phased, p.fh, p.p1, p.d1, p.s1, ry);
    const int slices = ax.n * ay.n * p.kchunks;
    const int kps = phased ? (slices + p.nsplit - 1) / p.nsplit : (int)p.ksteps_per_split;
    const int q0 = split * kps, q1 = min(q0 + kps, slices);
    const int cols = PASS == P_FWD ? p.W : p.OW, rows = PASS == P_FWD ? p.H : p.OH;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = tid & (G - 1), lrow = tid / G;
    const int pixb = p.Rcp * E;                    // bytes of a pixel's channels

    int pX[NB], pY[NB], pBase[NB];
#pragma unroll
    for (int r = 0; r < NB; ++r) {
        const int q = n0 + r * RP + lrow;
        const unsigned qc = (unsigned)min(q, ncol - 1);
        const int n = (int)(qc / (unsigned)(gw * gh));
        const unsigned yx = qc - (unsigned)n * (gw * gh);
        const int y = (int)(yx / (unsigned)gw), x = (int)yx - y * gw;
        pX[r] = PASS == P_FWD ? x * p.s0 : x;
        pY[r] = q < ncol ? (PASS == P_FWD ? y * p.s1 : y) : -(1 << 30);
        pBase[r] = (int)(((unsigned)(n * rows + (PASS == P_FWD ? y * p.s1 : y)) * cols + pX[r]) * pixb);
    }

    // the lane's slice of the next stage to load: index, channel slice, tap
    int q, c, ti, tj;
    {
        q = q0 + grp / GPC;
        const int u = q / p.kchunks;
        c = q - u * p.kchunks;
        tj = ax.n > 0 ? u / ax.n : 0;
        ti = u - tj * ax.n;
    }
    // one stage on: CPS slices are dt taps and dc slices (dt: dj rows of taps and di)
    const int dt = CPS / p.kchunks, dc = CPS - dt * p.kchunks;
    const int dj = ax.n > 0 ? dt / ax.n : 0, di = dt - dj * ax.n;
    auto next = [&] {
        q += CPS;
        c += dc;
        ti += di;
        tj += dj;
        if (c >= p.kchunks) {
            c -= p.kchunks;
            ++ti;
        }
        if (ti >= ax.n) {
            ti -= ax.n;
            ++tj;
        }
    };
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(wp), (short)0, p.wp_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(act), (short)0, p.act_bytes, 0x00020000);
    struct Stage {
        uint4 a[NA], b[NB];
    };
    auto load = [&](Stage &s) {
        // Past the range the sign bit takes every offset out of the resource.
        // The mask is opaque to the compiler: as a condition it became a branch
        // around each load, with a wait for all loads in flight inside.
        unsigned past = q < q1 ? 0u : 0x80000000u;
        asm volatile("" : "+v"(past));
        const int cb = c * (32 * E) + (grp % GPC) * 16;
        const int t = (ay.i0 + tj * ay.is) * p.fw + ax.i0 + ti * ax.is;
        const int sx = ax.start + ti * ax.step, sy = ay.start + tj * ay.step;
        const unsigned woff = (unsigned)(t * (int)p.M + m0 + lrow) * (unsigned)pixb + cb;
#pragma unroll
        for (int r = 0; r < NA; ++r) {
            const unsigned off = (woff + (unsigned)(RP * r * pixb)) | past | (m0 + lrow + RP * r < (int)p.M ? 0u : 0x80000000u);
            s.a[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)off, 0, 0));
        }
        const unsigned soff = (unsigned)((sy * cols + sx) * pixb + cb);
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const bool in = (unsigned)(pX[r] + sx) < (unsigned)cols && (unsigned)(pY[r] + sy) < (unsigned)rows;
            unsigned off = (unsigned)pBase[r] + soff;
            off = in ? off : 0x80000000u;
            s.b[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(off | past), 0, 0));
        }
        next();
    };
    // the rows of a lane's loads agree in the bits that swizzle them
    const int slot = lrow * SB + ((grp ^ (lrow & (G - 1))) * 16);
    auto store = [&](const Stage &s, char *buf) {
#pragma unroll
        for (int r = 0; r < NA; ++r) *reinterpret_cast<uint4 *>(buf + slot + r * (RP * SB)) = s.a[r];
#pragma unroll
        for (int r = 0; r < NB; ++r) *reinterpret_cast<uint4 *>(buf + TM * SB + slot + r * (RP * SB)) = s.b[r];
    };
    const int wm = wave >> 1, wn = wave & 1;
    const int r16 = lane & 15, g4 = lane >> 4;
    f32x4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const char *fa0 = lds[0] + (wm * (TM / 2) + r16) * SB, *fb0 = lds[0] + (TM + wn * (TN / 2) + r16) * SB;
    // The operands are (pixels, weights): a lane's four results are four
    // consecutive pixels of one output channel.
    auto compute = [&](int buf) {
        const char *fa = fa0 + buf * (int)sizeof(lds[0]), *fb = fb0 + buf * (int)sizeof(lds[0]);
#pragma unroll
        for (int h = 0; h < SB / 64; ++h) {
            const int sw = ((4 * h + g4) ^ (r16 & (G - 1))) * 16;
            uint4 a[MI], b[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) a[i] = *reinterpret_cast<const uint4 *>(fa + i * (16 * SB) + sw);
#pragma unroll
            for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const uint4 *>(fb + j * (16 * SB) + sw);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    if constexpr (MODE == M_F32) {
                        const float4 x = __builtin_bit_cast(float4, b[j]), y = __builtin_bit_cast(float4, a[i]);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, y.x, acc[i][j], 0, 0, 0);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, y.y, acc[i][j], 0, 0, 0);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, y.z, acc[i][j], 0, 0, 0);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, y.w, acc[i][j], 0, 0, 0);
                    } else if constexpr (MODE == M_BF16) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b[j]),
                                                                            __builtin_bit_cast(bf16x8_t, a[i]),
                                                                            acc[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, b[j]),
                                                                           __builtin_bit_cast(f16x8_t, a[i]),
                                                                           acc[i][j], 0, 0, 0);
                    }
                }
        }
    };

    const int stages = q1 > q0 ? (q1 - q0 + CPS - 1) / CPS : 0;  // the same for every lane
    if (stages > 0) {
        // loads past the last stage read zeros and are never multiplied
        Stage st[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            load(st[d]);
            // the loads stay in stage order: the loop's waits count them
            __builtin_amdgcn_sched_barrier(0);
        }
        store(st[0], lds[0]);
        load(st[0]);
        __builtin_amdgcn_sched_barrier(0);
        for (int k = 0;;) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                // stage k is in buffer d & 1; the other one was last read in
                // stage k - 1, before this barrier
                __syncthreads();
                store(st[(d + 1) % DEPTH], lds[(d + 1) & 1]);
                load(st[(d + 1) % DEPTH]);
                compute(d & 1);
                // straight out: an exit through the loop's end would make its
                // first waits count the loads of this stage as the newest
                if (++k == stages) goto done;
            }
        }
    }
done:
    cl_store<TOut, PASS, TM, TN>(out, partial, acc, p, t0, wm, wn, r16, g4, lds[0]);
}

// ------------------------------------------------- FP32 in three BF16 parts
// An FP32 value is the sum of three bfloat16 values, x = x1 + x2 + x3 (each the
// rounding of what the ones before leave; eight significant bits each make the
// 24 of FP32). A product x*w is the sum of the six part products down to 2^-16
// of it, x1w1, x1w2, x2w1, x2w2, x1w3, x3w1; the ones left out are 2^-24 of it
// and below. The BF16 matrix cores form each part product exactly and add 32
// of them at a time in FP32, at 16 times the rate of the FP32 ones, so six
// passes take 3/8 of the time, and the sums see fewer roundings than 4-deep
// FP32 steps: errors against FP64 are a third
// of the FP32 kernels' (1.4e-7 against 4.3e-7 relative at 576 products per sum,
// 4.1e-8 against 9.5e-8 at 27).
// The parts hold every value below 2^32 (nn_x3_parts.hpp). The copies flag what
// their blocks hold; a tile that reads a huge value, an infinity or a NaN, or
// tiny values and no others (whose results stay the FP32 kernels' to the bit),
// puts the parts together again and multiplies in FP32 instead.
// Channel-last copies in parts: [..][slice][part][32 channels], zeros past the
// reduction channels; the first nbw workgroups the weights [RS][M], wper of them
// for each tile's rows, the others 64 pixels by one slice each. flags: one word
// per workgroup.
constexpr int X3_T = 64;  // output tile
__global__ __launch_bounds__(256) void nn_x3_copies(uint16_t *__restrict__ wp, const float *__restrict__ w,
                                                    NNParams p, int dgrad, int nbw, int wper,
                                                    uint16_t *__restrict__ dst, const float *__restrict__ src, int hw,
                                                    int Cd, int npix, unsigned *__restrict__ flags) {
    int flag = 0;
    if ((int)blockIdx.x < nbw) {
        const int Rc = dgrad ? p.K : p.C, M = (int)p.M;
        const int wt = (int)blockIdx.x / wper, m0 = wt * X3_T, rows = min(X3_T, M - m0);
        const unsigned total = (unsigned)(p.RS * rows) * (unsigned)p.Rcp;
        for (unsigned e = (blockIdx.x - wt * wper) * 256u + threadIdx.x; e < total; e += (unsigned)wper * 256u) {
            const unsigned q = e / (unsigned)p.Rcp;
            const int r = (int)(e - q * (unsigned)p.Rcp);
            const int t = (int)(q / (unsigned)rows), m = m0 + (int)q - t * rows;
            float v = 0.f;
            if (r < Rc) {
                const int k = dgrad ? r : m, c = dgrad ? m : r;
                v = w[((long long)k * p.C + c) * p.RS + (p.RS - 1 - t)];
            }
            flag |= x3_flag(v);
            uint16_t h[3];
            x3_parts(v, h);
            uint16_t *o = wp + ((long long)(t * M + m) * p.kchunks + (r >> 5)) * 96 + (r & 31);
#pragma unroll
            for (int k = 0; k < 3; ++k) o[32 * k] = h[k];
        }
    } else {
        __shared__ unsigned tile[3][64 * 17];
        flag = x3_copy_block(dst, src, (int)blockIdx.x - nbw, hw, Cd, npix, p.kchunks, tile);
    }
    flag = x3_block_flags(flag);
    if (threadIdx.x == 0) flags[blockIdx.x] = (unsigned)flag;
}

// As nn_clgemm, one 32-deep slice (three parts, 64 bytes each per row) per
// stage, one LDS buffer and 64 x 64 tiles: four workgroups per CU cover each
// other's loads, stores and barriers (a stage is 24 MFMAs per wave; the matrix
// cores are busy 40% of the time, 34% in the data gradient). x1w1 has accumulators of its own, so
// that the five small products, 2^-8 of it and below, are not rounded to its
// last place each time; the two are added at the end. 56x56x64x32 -> 128, 3x3:
// 114 us with the copies (14 us of them) against 139 us in nn_clgemm on the FP32
// matrix cores, its data gradient 134 (25) against 153; where every tile runs in
// FP32 (x and dy at 1e20 throughout), 283 and 305 us. Wider tiles (64 x 128: 117 us, 128 x
// 128: 112 and 190 us) lose in occupancy what they save in LDS reads; two LDS
// buffers with one barrier per stage cost a workgroup per CU (121 us).
template <int PASS>
__global__ __launch_bounds__(NT, 2) void nn_x3gemm(float *__restrict__ out, const uint16_t *__restrict__ act,
                                                   const uint16_t *__restrict__ wp, const unsigned *__restrict__ flags,
                                                   int nbw, int wper, float *__restrict__ partial, NNParams p) {
    constexpr int TM = X3_T, TN = X3_T;
    constexpr int NA = TM / 64, NB = TN / 64, MI = TM / 32, NJ = TN / 32;
    constexpr int PLANE = (TM + TN) * 64;
    __shared__ __attribute__((aligned(16))) char lds[3 * PLANE];

    const ClTile t0 = cl_tile<PASS, TM, TN>(p);
    const int m0 = t0.m0, n0 = t0.n0, gw = t0.gw, gh = t0.gh, ncol = t0.ncol;
    if (n0 >= ncol) return;  // a phase's padding
    const TapAxis ax = tap_axis(PASS == P_FWD, t0.phased, p.fw, p.p0, p.d0, p.s0, t0.rx);
    const TapAxis ay = tap_axis(PASS == P_FWD, t0.phased, p.fh, p.p1, p.d1, p.s1, t0.ry);
    const int slices = ax.n * ay.n * p.kchunks;
    const int kps = t0.phased ? (slices + p.nsplit - 1) / p.nsplit : (int)p.ksteps_per_split;
    const int q0 = t0.split * kps, q1 = min(q0 + kps, slices);
    const int cols = PASS == P_FWD ? p.W : p.OW, rows = PASS == P_FWD ? p.H : p.OH;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = tid & 3, lrow = tid >> 2;  // 64 rows per load of the workgroup
    const int pixb = p.kchunks * 192;

    // the flags of what the tile reads: its rows' weights, and the pixel blocks
    // from its first row's first tap to its last row's last
    int flag = 0;
    {
        const int per = gw * gh, c1 = min(n0 + TN, ncol) - 1;
        const int na = n0 / per, nb = c1 / per;
        const int ya = (n0 - na * per) / gw, yb = (c1 - nb * per) / gw, s1 = PASS == P_FWD ? p.s1 : 1;
        const int ye = ay.start + (ay.n - 1) * ay.step;
        const int lo = (na * rows + min(max(ya * s1 + min(ay.start, ye), 0), rows - 1)) * cols;
        const int hi = (nb * rows + min(max(yb * s1 + max(ay.start, ye), 0), rows - 1)) * cols + cols - 1;
        const int wt = m0 / X3_T;
        for (int f = wt * wper + tid; f < (wt + 1) * wper; f += NT) flag |= (int)flags[f] & X3_HUGE;
        const int f1 = nbw + (hi / 64 + 1) * p.kchunks;
        for (int f = nbw + lo / 64 * p.kchunks + tid; f < f1; f += NT) flag |= (int)flags[f];
    }

    int pX[NB], pY[NB];
    unsigned pBase[NB];
#pragma unroll
    for (int r = 0; r < NB; ++r) {
        const int q = n0 + r * 64 + lrow;
        const unsigned qc = (unsigned)min(q, ncol - 1);
        const int n = (int)(qc / (unsigned)(gw * gh));
        const unsigned yx = qc - (unsigned)n * (gw * gh);
        const int y = (int)(yx / (unsigned)gw), x = (int)yx - y * gw;
        pX[r] = PASS == P_FWD ? x * p.s0 : x;
        pY[r] = q < ncol ? (PASS == P_FWD ? y * p.s1 : y) : -(1 << 30);
        pBase[r] = ((unsigned)(n * rows + (PASS == P_FWD ? y * p.s1 : y)) * cols + pX[r]) * pixb + grp * 16;
    }
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(wp), (short)0, p.wp_bytes, 0x00020000);
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(act), (short)0, p.act_bytes, 0x00020000);
    // the walk over (tap, slice), the same for every lane
    int q = q0, c, ti, tj;
    {
        const int u = q / p.kchunks;
        c = q - u * p.kchunks;
        tj = ax.n > 0 ? u / ax.n : 0;
        ti = u - tj * ax.n;
    }
    uint4 sa[NA][3], sb[NB][3];
    auto load = [&] {
        unsigned past = q < q1 ? 0u : 0x80000000u;  // opaque: no branch around the loads
        asm volatile("" : "+s"(past));
        const int t = (ay.i0 + tj * ay.is) * p.fw + ax.i0 + ti * ax.is;
        const int sx = ax.start + ti * ax.step, sy = ay.start + tj * ay.step;
        const unsigned woff = (unsigned)(t * (int)p.M + m0 + lrow) * (unsigned)pixb + c * 192 + grp * 16;
#pragma unroll
        for (int r = 0; r < NA; ++r) {
            const unsigned off = (woff + (unsigned)(64 * r * pixb)) | past | (m0 + lrow + 64 * r < (int)p.M ? 0u : 0x80000000u);
#pragma unroll
            for (int h = 0; h < 3; ++h)
                sa[r][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(off + 64 * h), 0, 0));
        }
        const unsigned soff = (unsigned)((sy * cols + sx) * pixb + c * 192);
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const bool in = (unsigned)(pX[r] + sx) < (unsigned)cols && (unsigned)(pY[r] + sy) < (unsigned)rows;
            unsigned off = pBase[r] + soff;
            off = (in ? off : 0x80000000u) | past;
#pragma unroll
            for (int h = 0; h < 3; ++h)
                sb[r][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(off + 64 * h), 0, 0));
        }
        ++q;
        if (++c == p.kchunks) {
            c = 0;
            if (++ti == ax.n) {
                ti = 0;
                ++tj;
            }
        }
    };
    // 64-byte rows, their groups XORed by the row pair
    char *slot = lds + lrow * 64 + ((grp ^ (lrow >> 1 & 3)) * 16);
    const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, g4 = lane >> 4;
    const int sw = (g4 ^ (r16 >> 1 & 3)) * 16;
    const char *fa = lds + (wm * (TM / 2) + r16) * 64 + sw, *fb = lds + (TM + wn * (TN / 2) + r16) * 64 + sw;
    f32x4_t acc[MI][NJ], low[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = low[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // parts to LDS, the next stage's loads
    auto stage = [&] {
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 3; ++h) {
#pragma unroll
            for (int r = 0; r < NA; ++r) *reinterpret_cast<uint4 *>(slot + h * PLANE + r * 4096) = sa[r][h];
#pragma unroll
            for (int r = 0; r < NB; ++r) *reinterpret_cast<uint4 *>(slot + h * PLANE + TM * 64 + r * 4096) = sb[r][h];
        }
        load();
        __syncthreads();
    };
    load();
    flag = x3_block_flags(flag);
    const bool fp32 = (flag & X3_HUGE) || (flag & (X3_TINY | X3_PLAIN)) == X3_TINY;
    for (int k = fp32 ? q1 : q0; k < q1; ++k) {
        stage();
        bf16x8_t a[MI][3];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int h = 0; h < 3; ++h) a[i][h] = *reinterpret_cast<const bf16x8_t *>(fa + h * PLANE + i * 1024);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            bf16x8_t b[3];
#pragma unroll
            for (int h = 0; h < 3; ++h) b[h] = *reinterpret_cast<const bf16x8_t *>(fb + h * PLANE + j * 1024);
            // the smallest products first
            constexpr int PB[5] = {2, 0, 1, 1, 0}, PA[5] = {0, 2, 1, 0, 1};
#pragma unroll
            for (int i = 0; i < MI; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[i][0], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 5; ++t)
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[PB[t]], a[i][PA[t]], low[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (acc[i][j] + low[i][j]) * X3_UNSCALE;
    if (fp32) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int k = q0; k < q1; ++k) {
            stage();
            // channels in the order of the FP32 kernels, 4 g4 + e of each half
            // slice; a pair at a time, for the registers
#pragma unroll 1
            for (int h = 0; h < 4; ++h) {
                const int at = (((h & 2) + (g4 >> 1)) ^ (r16 >> 1 & 3)) * 16 + (g4 & 1) * 8 + (h & 1) * 4 - sw;
                auto pair = [&](const char *row, float (&v)[2]) {
                    const unsigned a = *reinterpret_cast<const unsigned *>(row + at),
                                   b = *reinterpret_cast<const unsigned *>(row + at + PLANE),
                                   c = *reinterpret_cast<const unsigned *>(row + at + 2 * PLANE);
                    v[0] = x3_value(a & 0xffff, b & 0xffff, c & 0xffff);
                    v[1] = x3_value(a >> 16, b >> 16, c >> 16);
                };
                float a[MI][2], b[NJ][2];
#pragma unroll
                for (int i = 0; i < MI; ++i) pair(fa + i * 1024, a[i]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) pair(fb + j * 1024, b[j]);
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int i = 0; i < MI; ++i)
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][e], a[i][e], acc[i][j], 0, 0, 0);
            }
        }
    }
    cl_store<float, PASS, TM, TN>(out, partial, acc, p, t0, wm, wn, r16, g4, lds);
}

// ------------------------------------------------------------- kernel
template <int MODE, typename TIn, typename TOut, int PASS>
__global__ __launch_bounds__(NT) void nn_gemm(TOut *__restrict__ out, const TIn *__restrict__ in0,
                                              const TIn *__restrict__ in1, float *__restrict__ partial,
                                              NNParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char *tA = smem;
    char *tB = smem + Lds<MODE>::BYTES / 2;

    // Tile order: along Ncol fastest so concurrent workgroups share A rows.
    const long long tiles = p.tilesM * p.tilesN;
    const long long bid = blockIdx.x;
    const long long split = bid / tiles;
    const long long tl = bid - split * tiles;
    const long long tm = tl / p.tilesN, tn = tl - tm * p.tilesN;
    const long long m0 = tm * BM;
    // phased data gradient: the tile's phase and its column offset in it
    int ph = 0;
    long long n0 = tn * BN;
    long long ksteps = p.ksteps, kps = p.ksteps_per_split;
    if (PASS == P_DGRAD && p.phased) {
        while (ph + 1 < p.nph && tn >= p.ph_tile0[ph + 1]) ++ph;
        n0 = (tn - p.ph_tile0[ph]) * BN;
        const int rx = ph % p.s0, ry = ph / p.s0;
        ksteps = (long long)phase_taps(p.fw, rx, p.p0, p.d0, p.s0) * phase_taps(p.fh, ry, p.p1, p.d1, p.s1) *
                 p.kchunks;
        kps = (ksteps + p.nsplit - 1) / p.nsplit;
    }

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = tid & 127, kk0 = (tid >> 7) * 16;

    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const long long ks0 = split * kps;
    long long ks1 = ks0 + kps;
    if (ks1 > ksteps) ks1 = ksteps;

    {
        Gather<TIn, PASS> g(in0, in1, p, m0 + lrow, n0 + lrow, ph);
        float va[16], vb[16];
        if (ks0 < ks1) g.load(ks0, kk0, va, vb);
        for (long long ks = ks0; ks < ks1; ++ks) {
            __syncthreads();
            store_row16<MODE>(tA, lrow, kk0, va);
            store_row16<MODE>(tB, lrow, kk0, vb);
            __syncthreads();
            if (ks + 1 < ks1) g.load(ks + 1, kk0, va, vb);
            mma_slice<MODE>(tA, tB, wm, wn, lane, acc);
        }
    }

    // Epilogue. acc[i][j][v] is C[row][col] with
    // row = m0 + wm*64 + i*16 + 4*(lane/16) + v, col = n0 + wn*64 + j*16 + lane%16.
    // Split reductions store FP32 partial tiles (row-major over the padded
    // columns; nn_split_reduce / wgrad_reduce sum them in split order).
    const int g4 = (lane >> 4) * 4, c16 = lane & 15;
    if (p.nsplit > 1) {
        const long long pc0 = (PASS == P_DGRAD && p.phased) ? (long long)p.ph_tile0[ph] * BN : 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const long long col = n0 + wn * 64 + j * 16 + c16;
            if (pc0 + col >= p.Ncol) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const long long row = m0 + wm * 64 + i * 16 + g4 + v;
                    if (row < p.M) partial[(split * p.M + row) * p.Ncol + pc0 + col] = acc[i][j][v];
                }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const long long col = n0 + wn * 64 + j * 16 + c16;
        long long cbase;
        long long rstride;
        if constexpr (PASS == P_FWD) {
            if (col >= p.Ncol) continue;
            const Pix q = decode(col, p.OH, p.OW);
            const long long ohw = (long long)p.OH * p.OW;
            cbase = (long long)q.n * p.K * ohw + (long long)q.a * p.OW + q.b;
            rstride = ohw;
        } else if constexpr (PASS == P_DGRAD) {
            const long long hw = (long long)p.H * p.W;
            if (p.phased) {
                const int rx = ph % p.s0, ry = ph / p.s0;
                const int Mx = phase_len(p.W, p.s0, rx), My = phase_len(p.H, p.s1, ry);
                if (col >= (long long)p.N * My * Mx) continue;
                const Pix q = decode(col, My, Mx);
                cbase = (long long)q.n * p.C * hw + (long long)(p.s1 * q.a + ry) * p.W + (p.s0 * q.b + rx);
            } else {
                if (col >= p.Ncol) continue;
                const Pix q = decode(col, p.H, p.W);
                cbase = (long long)q.n * p.C * hw + (long long)q.a * p.W + q.b;
            }
            rstride = hw;
        } else {
            if (col >= p.Ncol) continue;
            // dW[fw-1-i, fh-1-j, c, k]: element (k*C + c)*RS + RS-1-t
            const int c = (int)(col / p.RS);
            const int t = (int)(col - (long long)c * p.RS);
            cbase = (long long)c * p.RS + (p.RS - 1 - t);
            rstride = (long long)p.C * p.RS;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const long long row = m0 + wm * 64 + i * 16 + g4 + v;
                if (row >= p.M) continue;
                st_f(out, cbase + row * rstride, acc[i][j][v]);
            }
    }
}

// Second stage of a split forward or data gradient: sums the nsplit partial
// tiles of each output element in split order (deterministic) and stores it
// in the output layout. Padding columns of the phased layout are skipped.
// blockIdx.y: output channel; a lane owns columns, 32-bit throughout (the
// launcher keeps M * Ncol of a split problem below 2^26).
template <typename TOut, int PASS>
__global__ __launch_bounds__(256) void nn_split_reduce(TOut *__restrict__ out, const float *__restrict__ partial,
                                                       NNParams p) {
    const int row = blockIdx.y, nall = (int)p.Ncol;
    const long long total = p.M * p.Ncol;
    const float *src = partial + (long long)row * nall;
    for (int col = blockIdx.x * 256 + threadIdx.x; col < nall; col += gridDim.x * 256) {
        long long dst;
        if constexpr (PASS == P_FWD) {
            const int ohw = p.OH * p.OW, n = col / ohw;
            dst = ((long long)n * p.K + row) * ohw + (col - n * ohw);
        } else {
            const int hw = p.H * p.W;
            if (p.phased) {
                const int tn = col / BN;
                int ph = 0;
                while (ph + 1 < p.nph && tn >= p.ph_tile0[ph + 1]) ++ph;
                const int lc = col - p.ph_tile0[ph] * BN;
                const int rx = ph % p.s0, ry = ph / p.s0;
                const int Mx = phase_len(p.W, p.s0, rx), My = phase_len(p.H, p.s1, ry);
                if (lc >= p.N * My * Mx) continue;
                const int n = lc / (My * Mx), yx = lc - n * (My * Mx), y = yx / Mx, x = yx - y * Mx;
                dst = ((long long)n * p.C + row) * hw + (long long)(p.s1 * y + ry) * p.W + (p.s0 * x + rx);
            } else {
                const int n = col / hw;
                dst = ((long long)n * p.C + row) * hw + (col - n * hw);
            }
        }
        float s = 0.f;
        int sp = 0;
        for (; sp + 4 <= p.nsplit; sp += 4) {  // four loads in flight, summed in split order
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = src[(sp + k) * total + col];
#pragma unroll
            for (int k = 0; k < 4; ++k) s += v[k];
        }
        for (; sp < p.nsplit; ++sp) s += src[sp * total + col];
        st_f(out, dst, s);
    }
}

// Deterministic second stage of the split filter gradient: sums the nsplit
// partial tiles in split order and scatters into dW's layout.
template <typename TOut>
__global__ __launch_bounds__(256) void wgrad_reduce(TOut *__restrict__ out,
                                                    const float *__restrict__ partial,
                                                    NNParams p) {
    const long long total = p.M * p.Ncol;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        float s = 0.f;
        for (int sp = 0; sp < p.nsplit; ++sp) s += partial[sp * total + e];
        const long long row = e / p.Ncol, col = e - row * p.Ncol;
        const int c = (int)(col / p.RS);
        const int t = (int)(col - (long long)c * p.RS);
        st_f(out, row * ((long long)p.C * p.RS) + (long long)c * p.RS + (p.RS - 1 - t), s);
    }
}

// ------------------------------------------------------------- host side
static int setup(NNParams &p, int pass, const long long *xd, const long long *wd,
                 const long long *yd, const long long *st, const long long *pd,
                 const long long *dl) {
    p.W = (int)xd[0];
    p.H = (int)xd[1];
    p.C = (int)xd[2];
    p.N = (int)xd[3];
    p.fw = (int)wd[0];
    p.fh = (int)wd[1];
    p.K = (int)wd[3];
    p.OW = (int)yd[0];
    p.OH = (int)yd[1];
    p.s0 = (int)st[0];
    p.s1 = (int)st[1];
    p.p0 = (int)pd[0];
    p.p1 = (int)pd[1];
    p.d0 = (int)dl[0];
    p.d1 = (int)dl[1];
    if (wd[2] != xd[2] || yd[2] != wd[3] || yd[3] != xd[3]) return K_ERR_SIZE;
    if (p.s0 < 1 || p.s1 < 1 || p.d0 < 1 || p.d1 < 1) return K_ERR_ARG;
    p.RS = p.fw * p.fh;
    p.nsplit = 1;
    p.phased = 0;
    p.nph = 1;
    p.cl = 0;
    p.Rcp = 0;
    p.wp_bytes = p.act_bytes = 0;
    p.nsplit_req = 0;
    for (int i = 0; i <= kMaxPhases; ++i) p.ph_tile0[i] = 0;
    if (pass == P_FWD) {
        p.M = p.K;
        p.Ncol = (long long)p.N * p.OH * p.OW;
        p.kchunks = (p.C + BK - 1) / BK;
        p.ksteps = (long long)p.RS * p.kchunks;
    } else if (pass == P_DGRAD) {
        p.M = p.C;
        p.Ncol = (long long)p.N * p.H * p.W;
        p.kchunks = (p.K + BK - 1) / BK;
        p.ksteps = (long long)p.RS * p.kchunks;
        // AFHIP_NN_PHASED=0 in the environment keeps the unphased order
        const char *env = std::getenv("AFHIP_NN_PHASED");
        const bool off = env && env[0] == '0';
        if (!off && (p.s0 > 1 || p.s1 > 1) && p.s0 * p.s1 <= kMaxPhases) {
            p.phased = 1;
            p.nph = p.s0 * p.s1;
            long long t0 = 0, kmax = 0;
            for (int ph = 0; ph < p.nph; ++ph) {
                const int rx = ph % p.s0, ry = ph / p.s0;
                const long long cols = (long long)p.N * phase_len(p.H, p.s1, ry) * phase_len(p.W, p.s0, rx);
                p.ph_tile0[ph] = (int)t0;
                t0 += (cols + BN - 1) / BN;
                const long long ks = (long long)phase_taps(p.fw, rx, p.p0, p.d0, p.s0) *
                                     phase_taps(p.fh, ry, p.p1, p.d1, p.s1) * p.kchunks;
                if (ks > kmax) kmax = ks;
            }
            if (t0 >= (1LL << 31)) return K_ERR_SIZE;
            p.ph_tile0[p.nph] = (int)t0;
            p.Ncol = t0 * BN;
            p.ksteps = kmax;
        }
    } else {
        p.M = p.K;
        p.Ncol = (long long)p.C * p.RS;
        p.kchunks = 0;
        const long long R = (long long)p.N * p.OH * p.OW;
        p.ksteps = (R + BK - 1) / BK;
    }
    p.ksteps_per_split = p.ksteps;
    p.tilesM = (p.M + BM - 1) / BM;
    p.tilesN = (p.Ncol + BN - 1) / BN;
    return K_OK;
}

// Split count for the filter gradient: enough workgroups to cover the chip
// about twice, each with at least 16 slices of R.
static int wgrad_splits(const NNParams &p) {
    const long long tiles = p.tilesM * p.tilesN;
    long long want = (512 + tiles - 1) / tiles;
    long long maxs = p.ksteps / 16;
    if (want > maxs) want = maxs;
    if (want < 1) want = 1;
    return (int)want;
}

// The channel-last path runs when the operands are stored in the MMA's
// operand type (FP32, BF16 or FP16 arrays at their own precision).
template <int MODE, typename TIn>
constexpr bool cl_eligible() {
    return (MODE == M_F32 && std::is_same<TIn, float>::value) ||
           (MODE == M_BF16 && std::is_same<TIn, bf16s>::value) ||
           (MODE == M_F16 && std::is_same<TIn, _Float16>::value);
}

// Workspace of the forward / data-gradient GEMM: packed weights and the
// channel-last activation (esz > 0: element bytes of the channel-last path),
// then the split partials; every part 256-byte aligned.
// AFHIP_NN_CL=0 in the environment disables the channel-last path.
struct GemmLayout {
    int cl = 0, Rcp = 0, wp_bytes = 0, act_bytes = 0;
    long long off_w = 0, off_act = 0, off_part = 0, total = 0;
};
static GemmLayout gemm_layout(const NNParams &p, int pass, int esz, int nsplit) {
    GemmLayout L;
    auto al = [](long long b) { return (b + 255) & ~255LL; };
    const char *env = std::getenv("AFHIP_NN_CL");
    const long long Rcp = (long long)p.kchunks * BK;
    const long long rows = pass == P_FWD ? p.H : p.OH, cols = pass == P_FWD ? p.W : p.OW;
    const long long wb = (long long)p.RS * p.M * Rcp * esz, ab = (long long)p.N * rows * cols * Rcp * esz;
    // the copies are read through buffer resources (32-bit byte offsets)
    // and columns and rows counted in 32 bits
    if (esz > 0 && !(env && env[0] == '0') && wb < (1LL << 31) - 64 && ab < (1LL << 31) - 64 &&
        p.Ncol < (1LL << 30) && p.M < (1LL << 24) && (p.phased || pass == P_FWD || (p.s0 == 1 && p.s1 == 1))) {
        L.cl = 1;
        L.Rcp = (int)Rcp;
        L.wp_bytes = (int)wb;
        L.act_bytes = (int)ab;
        L.off_w = 0;
        L.off_act = al(wb);
        L.off_part = L.off_act + al(ab);
    }
    L.total = L.off_part + (nsplit > 1 ? (long long)nsplit * p.M * p.Ncol * 4 : 0);
    return L;
}

// Split count for the forward and data gradient: layers whose output tiles
// leave most CUs idle split the reduction (FP32 partial tiles, a second
// summing pass), about two workgroups per CU, each with at least 4 slices,
// the partials within 256 MiB. AFHIP_NN_SPLIT=<n> in the environment forces
// n (1 = unsplit).
static int gemm_splits(const NNParams &p) {
    const long long tiles = p.tilesM * p.tilesN;
    long long want;
    const char *env = std::getenv("AFHIP_NN_SPLIT");
    if (env && env[0] >= '1' && env[0] <= '9') {
        want = std::atoll(env);
    } else if (p.nsplit_req > 0) {
        want = p.nsplit_req;
    } else {
        const long long cus = cu_count_current();
        if (tiles * 2 >= cus) return 1;
        want = (2 * cus + tiles - 1) / tiles;
        const long long maxs = p.ksteps / 4;
        if (want > maxs) want = maxs;
    }
    while (want > 1 && want * p.M * p.Ncol * 4 > (256LL << 20)) --want;
    if (want > p.ksteps) want = p.ksteps;
    if (want < 1 || p.M > 65535) want = 1;  // the summing pass counts channels in gridDim.y
    return (int)want;
}

template <int MODE, typename TIn, typename TOut, int TM, int TN>
static void cl_launch_tile(int pass, TOut *out, const TIn *act, const TIn *wp, float *part, NNParams &p,
                           hipStream_t s) {
    p.tilesM = (p.M + TM - 1) / TM;
    p.tilesN = (p.Ncol + TN - 1) / TN;
    auto fn = pass == P_FWD ? nn_clgemm<MODE, TIn, TOut, P_FWD, TM, TN> : nn_clgemm<MODE, TIn, TOut, P_DGRAD, TM, TN>;
    fn<<<(unsigned)(p.tilesM * p.tilesN * p.nsplit), NT, 0, s>>>(out, act, wp, part, p);
}

// Wide tiles where they give at least half of the CUs a workgroup, 64 x 64
// below that (28x28x128x32 -> 128, BF16, 196 wide tiles: 24 us against 29;
// 14x14x256x32 -> 256, 98 wide tiles: 35 us against 31), and for FP32 at any
// size: its 64 x 64 tiles keep three or four workgroups per CU to cover the
// stages' loads, the wide ones two (56x56x64x32 -> 128: 139 us against 164).
// 64 rows where 128 would leave half of the last tile empty.
template <int MODE, typename TIn, typename TOut>
static void cl_launch(int pass, TOut *out, const TIn *act, const TIn *wp, float *part, NNParams &p, hipStream_t s) {
    const bool half = (p.M - 1) % 128 < 64;
    const long long wide = (half ? (p.M + 63) / 64 : (p.M + 127) / 128) * ((p.Ncol + 127) / 128) * p.nsplit;
    if (MODE == M_F32 || 2 * wide < cu_count_current())
        cl_launch_tile<MODE, TIn, TOut, 64, 64>(pass, out, act, wp, part, p, s);
    else if constexpr (MODE != M_F32) {
        if (half)
            cl_launch_tile<MODE, TIn, TOut, 64, 128>(pass, out, act, wp, part, p, s);
        else
            cl_launch_tile<MODE, TIn, TOut, 128, 128>(pass, out, act, wp, part, p, s);
    }
}

template <int MODE, typename TIn, typename TOut>
static int run(int pass, void *out, const void *a0, const void *a1, NNParams &p, void *ws,
               long long ws_bytes, hipStream_t s) {
    if (p.M == 0 || p.Ncol == 0) return K_OK;
    const int smem = Lds<MODE>::BYTES;
    const long long tiles = p.tilesM * p.tilesN;
    if (pass == P_FWD || pass == P_DGRAD) {
        p.nsplit = gemm_splits(p);
        constexpr bool kCL = cl_eligible<MODE, TIn>();
        GemmLayout L = gemm_layout(p, pass, kCL ? (int)sizeof(TIn) : 0, p.nsplit);
        if (ws == nullptr || ws_bytes < L.total) {
            // a short workspace: drop the split, then the channel-last copies
            p.nsplit = 1;
            L = gemm_layout(p, pass, kCL ? (int)sizeof(TIn) : 0, 1);
            if (ws == nullptr || ws_bytes < L.total) L = gemm_layout(p, pass, 0, 1);
        }
        p.ksteps_per_split = (p.ksteps + p.nsplit - 1) / p.nsplit;
        char *wsb = (char *)ws;
        float *part = p.nsplit > 1 ? (float *)(wsb + L.off_part) : nullptr;
        const unsigned grid = (unsigned)(tiles * p.nsplit);
        if constexpr (kCL) {
            if (L.cl) {
                p.cl = 1;
                p.Rcp = L.Rcp;
                p.wp_bytes = L.wp_bytes;
                p.act_bytes = L.act_bytes;
                TIn *wp = (TIn *)(wsb + L.off_w), *act = (TIn *)(wsb + L.off_act);
                const long long nw = (long long)p.RS * p.M * p.Rcp;
                const long long b1 = std::min<long long>((nw + 255) / 256, 4096);
                const int rows = pass == P_FWD ? p.H : p.OH, cols = pass == P_FWD ? p.W : p.OW;
                const int Cd = pass == P_FWD ? p.C : p.K;
                const int npix = p.N * rows * cols;  // below 2^31 / Rcp
                const int ncg = (p.Rcp * (int)sizeof(TIn) + 127) / 128;
                const long long b2 = (long long)((npix + 63) / 64) * ncg;
                nn_cl_copies<TIn><<<(unsigned)(b1 + b2), 256, 0, s>>>(wp, (const TIn *)a1, p, pass == P_DGRAD,
                                                                      (int)b1, act, (const TIn *)a0, rows * cols, Cd,
                                                                      npix, ncg);
                cl_launch<MODE, TIn, TOut>(pass, (TOut *)out, act, wp, part, p, s);
            }
        }
        if (!p.cl) {
            auto fn = pass == P_FWD ? nn_gemm<MODE, TIn, TOut, P_FWD> : nn_gemm<MODE, TIn, TOut, P_DGRAD>;
            fn<<<grid, NT, smem, s>>>((TOut *)out, (const TIn *)a0, (const TIn *)a1, part, p);
        }
        if (p.nsplit > 1) {
            auto red = pass == P_FWD ? nn_split_reduce<TOut, P_FWD> : nn_split_reduce<TOut, P_DGRAD>;
            red<<<dim3((unsigned)((p.Ncol + 255) / 256), (unsigned)p.M), 256, 0, s>>>((TOut *)out, part, p);
        }
    } else {
        if (p.ksteps == 0) {
            // empty reduction: dW = 0
            return afhip_k_fill(sizeof(TOut) == 4 ? DT_F32 : (std::is_same<TOut, bf16s>::value ? DT_BF16 : DT_F16),
                                out, 0.0, p.M * p.Ncol, s);
        }
        p.nsplit = wgrad_splits(p);
        const long long need = (long long)p.nsplit * p.M * p.Ncol * 4;
        if (p.nsplit > 1 && (ws == nullptr || ws_bytes < need)) p.nsplit = 1;
        p.ksteps_per_split = (p.ksteps + p.nsplit - 1) / p.nsplit;
        p.nsplit = (int)((p.ksteps + p.ksteps_per_split - 1) / p.ksteps_per_split);
        nn_gemm<MODE, TIn, TOut, P_WGRAD><<<dim3((unsigned)(tiles * p.nsplit)), NT, smem, s>>>(
            (TOut *)out, (const TIn *)a0, (const TIn *)a1, (float *)ws, p);
        if (p.nsplit > 1) {
            long long blocks = (p.M * p.Ncol + 255) / 256;
            if (blocks > kMaxGridBlocks) blocks = kMaxGridBlocks;
            wgrad_reduce<TOut><<<dim3((unsigned)blocks), 256, 0, s>>>((TOut *)out, (const float *)ws, p);
        }
    }
    return launch_status();
}

static int dispatch(int pass, int in_type, int out_type, int precision, void *out,
                    const void *a0, const void *a1, NNParams &p, void *ws, long long wsb,
                    hipStream_t s) {
    // precision: 0 default, 1 bf16, 2 f16, 3 split, 4 f32 (afhip_precision)
    int mode;
    switch (precision) {
        case 0:
            mode = in_type == DT_F32 ? M_F32 : in_type == DT_BF16 ? M_BF16 : in_type == DT_F16 ? M_F16 : -1;
            break;
        case 1: mode = M_BF16; break;
        case 2: mode = M_F16; break;
        case 3: mode = M_SPLIT; break;
        case 4: mode = M_F32; break;
        default: return K_ERR_ARG;
    }
    if (mode < 0) return K_ERR_TYPE;
#define GO(MD, TI, TO) return run<MD, TI, TO>(pass, out, a0, a1, p, ws, wsb, s)
    if (in_type == DT_F32) {
        if (out_type != DT_F32) return K_ERR_TYPE;
        switch (mode) {
            case M_F32: GO(M_F32, float, float);
            case M_BF16: GO(M_BF16, float, float);
            case M_F16: GO(M_F16, float, float);
            case M_SPLIT: GO(M_SPLIT, float, float);
        }
    } else if (in_type == DT_BF16) {
        if (mode != M_BF16) return K_ERR_TYPE;
        if (out_type == DT_F32) GO(M_BF16, bf16s, float);
        if (out_type == DT_BF16) GO(M_BF16, bf16s, bf16s);
    } else if (in_type == DT_F16) {
        if (mode != M_F16) return K_ERR_TYPE;
        if (out_type == DT_F32) GO(M_F16, _Float16, float);
        if (out_type == DT_F16) GO(M_F16, _Float16, _Float16);
    }
#undef GO
    return K_ERR_TYPE;
}

// ---- FP32 in three BF16 parts
struct X3Layout {
    int wp_bytes = 0, act_bytes = 0, wper = 0, nbw = 0, nba = 0, npix = 0;
    long long off_act = 0, off_flag = 0, off_part = 0, total = 0;
};
static bool x3_layout(const NNParams &p, int pass, X3Layout *L) {
    auto al = [](long long b) { return (b + 255) & ~255LL; };
    const long long rows = pass == P_FWD ? p.H : p.OH, cols = pass == P_FWD ? p.W : p.OW;
    const long long wb = (long long)p.RS * p.M * p.kchunks * 192, npix = (long long)p.N * rows * cols;
    const long long ab = npix * p.kchunks * 192;
    // an activation without pixels (outputs of padding alone) has no flags to read
    if (npix < 1) return false;
    // offsets past a resource's end must not wrap
    if (wb >= (1LL << 30) || ab >= (1LL << 30) || p.Ncol >= (1LL << 30) || p.M >= (1LL << 24)) return false;
    if (pass == P_DGRAD && !p.phased && (p.s0 > 1 || p.s1 > 1)) return false;
    L->wp_bytes = (int)wb;
    L->act_bytes = (int)ab;
    L->npix = (int)npix;
    // weight blocks: a lane per element of a tile's rows, about a thousand in all
    const long long wt = (p.M + X3_T - 1) / X3_T, each = (long long)p.RS * X3_T * p.kchunks * BK;
    L->wper = (int)std::max<long long>(1, std::min<long long>((each + 255) / 256, 1024 / wt));
    L->nbw = (int)wt * L->wper;
    L->nba = (int)((npix + 63) / 64 * p.kchunks);
    L->off_act = al(wb);
    L->off_flag = L->off_act + al(ab);
    L->off_part = L->off_flag + al(4LL * (L->nbw + L->nba));
    L->total = L->off_part + (p.nsplit > 1 ? (long long)p.nsplit * p.M * p.Ncol * 4 : 0);
    return true;
}

static int x3_setup(NNParams &p, X3Layout *L, int pass, const long long *xd, const long long *wd, const long long *yd,
                    const long long *st, const long long *pd, const long long *dl, int nsplit) {
    if (pass != P_FWD && pass != P_DGRAD) return K_ERR_ARG;
    const int rc = setup(p, pass, xd, wd, yd, st, pd, dl);
    if (rc) return rc;
    if (p.M == 0 || p.Ncol == 0 || p.kchunks == 0) return K_ERR_NOT_SUPPORTED;
    p.nsplit_req = nsplit > 0 ? nsplit : 1;
    p.nsplit = gemm_splits(p);
    p.ksteps_per_split = (p.ksteps + p.nsplit - 1) / p.nsplit;
    p.Rcp = p.kchunks * BK;
    return x3_layout(p, pass, L) ? K_OK : K_ERR_NOT_SUPPORTED;
}

long long nn_x3_workspace(int pass, const long long *xd, const long long *wd, const long long *yd,
                          const long long *st, const long long *pd, const long long *dl, int nsplit) {
    NNParams p;
    X3Layout L;
    return x3_setup(p, &L, pass, xd, wd, yd, st, pd, dl, nsplit) == K_OK ? L.total : 0;
}

int nn_x3(int pass, void *out, const void *in, const void *w, const long long *xd, const long long *wd,
          const long long *yd, const long long *st, const long long *pd, const long long *dl, int nsplit, void *ws,
          long long ws_bytes, hipStream_t s) {
    NNParams p;
    X3Layout L;
    const int rc = x3_setup(p, &L, pass, xd, wd, yd, st, pd, dl, nsplit);
    if (rc) return rc;
    if (ws == nullptr || ws_bytes < L.total) return K_ERR_ARG;
    char *b = (char *)ws;
    uint16_t *wp = (uint16_t *)b, *act = (uint16_t *)(b + L.off_act);
    unsigned *flags = (unsigned *)(b + L.off_flag);
    float *part = p.nsplit > 1 ? (float *)(b + L.off_part) : nullptr;
    p.wp_bytes = L.wp_bytes;
    p.act_bytes = L.act_bytes;
    const int rows = pass == P_FWD ? p.H : p.OH, cols = pass == P_FWD ? p.W : p.OW;
    nn_x3_copies<<<(unsigned)(L.nbw + L.nba), 256, 0, s>>>(wp, (const float *)w, p, pass == P_DGRAD, L.nbw, L.wper,
                                                          act, (const float *)in, rows * cols,
                                                          pass == P_FWD ? p.C : p.K, L.npix, flags);
    p.tilesM = (p.M + X3_T - 1) / X3_T;
    p.tilesN = (p.Ncol + X3_T - 1) / X3_T;
    auto fn = pass == P_FWD ? nn_x3gemm<P_FWD> : nn_x3gemm<P_DGRAD>;
    fn<<<(unsigned)(p.tilesM * p.tilesN * p.nsplit), NT, 0, s>>>((float *)out, act, wp, flags, L.nbw, L.wper,
                                                                 part, p);
    if (p.nsplit > 1) {
        auto red = pass == P_FWD ? nn_split_reduce<float, P_FWD> : nn_split_reduce<float, P_DGRAD>;
        red<<<dim3((unsigned)((p.Ncol + 255) / 256), (unsigned)p.M), 256, 0, s>>>((float *)out, part, p);
    }
    return launch_status();
}

}  // namespace afhip

using namespace afhip;

extern "C" long long afhip_k_conv2_nn_gemm_split_workspace(int pass, int in_type, int precision,
                                                           const long long *xdims, const long long *wdims,
                                                           const long long *ydims, const long long *stride,
                                                           const long long *pad, const long long *dil,
                                                           int nsplit) {
    if (pass != P_FWD && pass != P_DGRAD) return 0;
    NNParams p;
    if (setup(p, pass, xdims, wdims, ydims, stride, pad, dil)) return 0;
    if (p.M == 0 || p.Ncol == 0) return 0;
    p.nsplit_req = nsplit > 0 ? nsplit : 0;
    // channel-last path: operands stored at their own precision
    const bool cl = (in_type == DT_F32 && (precision == 0 || precision == 4)) ||
                    (in_type == DT_BF16 && (precision == 0 || precision == 1)) ||
                    (in_type == DT_F16 && (precision == 0 || precision == 2));
    const int esz = cl ? (in_type == DT_F32 ? 4 : 2) : 0;
    return gemm_layout(p, pass, esz, gemm_splits(p)).total;
}

extern "C" int afhip_k_conv2_nn_gemm_split(int pass, int in_type, int out_type, int precision, void *out,
                                           const void *in, const void *w, const long long *xdims,
                                           const long long *wdims, const long long *ydims,
                                           const long long *stride, const long long *pad, const long long *dil,
                                           int nsplit, void *workspace, long long workspace_bytes, void *stream) {
    if (pass != P_FWD && pass != P_DGRAD) return K_ERR_ARG;
    NNParams p;
    int rc = setup(p, pass, xdims, wdims, ydims, stride, pad, dil);
    if (rc) return rc;
    p.nsplit_req = nsplit > 0 ? nsplit : 0;
    return dispatch(pass, in_type, out_type, precision, out, in, w, p, workspace, workspace_bytes,
                    (hipStream_t)stream);
}

extern "C" long long afhip_k_conv2_nn_gemm_workspace(int pass, int in_type, int precision, const long long *xdims,
                                                     const long long *wdims, const long long *ydims,
                                                     const long long *stride, const long long *pad,
                                                     const long long *dil) {
    return afhip_k_conv2_nn_gemm_split_workspace(pass, in_type, precision, xdims, wdims, ydims, stride, pad, dil,
                                                 0);
}

extern "C" int afhip_k_conv2_nn_gemm(int pass, int in_type, int out_type, int precision, void *out,
                                     const void *in, const void *w, const long long *xdims,
                                     const long long *wdims, const long long *ydims,
                                     const long long *stride, const long long *pad, const long long *dil,
                                     void *workspace, long long workspace_bytes, void *stream) {
    return afhip_k_conv2_nn_gemm_split(pass, in_type, out_type, precision, out, in, w, xdims, wdims, ydims, stride,
                                       pad, dil, 0, workspace, workspace_bytes, stream);
}

extern "C" int afhip_k_conv2_nn_fwd(int in_type, int out_type, int precision, void *y,
                                    const void *x, const void *w, const long long *xdims,
                                    const long long *wdims, const long long *ydims,
                                    const long long *stride, const long long *pad,
                                    const long long *dil, void *stream) {
    return afhip_k_conv2_nn_gemm(P_FWD, in_type, out_type, precision, y, x, w, xdims, wdims, ydims, stride, pad,
                                 dil, nullptr, 0, stream);
}

extern "C" int afhip_k_conv2_nn_dgrad(int in_type, int out_type, int precision, void *dx,
                                      const void *dy, const void *w, const long long *xdims,
                                      const long long *wdims, const long long *ydims,
                                      const long long *stride, const long long *pad,
                                      const long long *dil, void *stream) {
    return afhip_k_conv2_nn_gemm(P_DGRAD, in_type, out_type, precision, dx, dy, w, xdims, wdims, ydims, stride,
                                 pad, dil, nullptr, 0, stream);
}

extern "C" long long afhip_k_conv2_nn_wgrad_workspace(const long long *xdims, const long long *wdims,
                                                      const long long *ydims, const long long *stride,
                                                      const long long *pad, const long long *dil) {
    NNParams p;
    if (setup(p, P_WGRAD, xdims, wdims, ydims, stride, pad, dil)) return 0;
    const int ns = wgrad_splits(p);
    return ns > 1 ? (long long)ns * p.M * p.Ncol * 4 : 0;
}

extern "C" int afhip_k_conv2_nn_wgrad(int in_type, int out_type, int precision, void *dw,
                                      const void *x, const void *dy, const long long *xdims,
                                      const long long *wdims, const long long *ydims,
                                      const long long *stride, const long long *pad,
                                      const long long *dil, void *workspace,
                                      long long workspace_bytes, void *stream) {
    NNParams p;
    int rc = setup(p, P_WGRAD, xdims, wdims, ydims, stride, pad, dil);
    if (rc) return rc;
    return dispatch(P_WGRAD, in_type, out_type, precision, dw, x, dy, p, workspace, workspace_bytes,
                    (hipStream_t)stream);
}
