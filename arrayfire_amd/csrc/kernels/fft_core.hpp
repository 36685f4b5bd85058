// Register FFTs of power-of-two length for the frequency-domain convolution.
//
// A transform of L = 8^a * r points (r = 1, 2 or 4) is held by L / 8 lanes,
// eight values per lane: lane t holds points t + j * L/8. Stockham passes of
// radix 8 (the last of radix 2 or 4 when L is no power of 8) run in registers
// and exchange through LDS between passes, so a 2048-point transform crosses
// LDS three times where radix-2 stages cross it eleven times. Input and output
// are both in natural order and in the same lanes, so a product of two
// spectra needs no exchange at all. LDS rows are padded by one value in eight:
// without it the first pass writes 64 bytes apart, into four banks.
//
// Twiddles (computed in double, then rounded) come from a table laid out as
// the lanes read it, [twiddle][lane] per length, and are kept in registers: a
// kernel that runs several transforms loads them once. Gathered from one
// W_4096 table instead, the 20 loads of a 2048-point transform touch up to 64
// cache lines each, which cost more than the arithmetic.
#pragma once
#include "kcommon.hpp"

namespace afhip {

constexpr int FFT_LMAX = 4096;  // longest in-LDS transform

// W_4096^j, j < 2048, for the general passes
static __device__ float2 g_fft_tw32[FFT_LMAX / 2];
static __device__ double2 g_fft_tw64[FFT_LMAX / 2];

// RegFft<., LOGL>: radix-8 passes, radix of the last pass (1: none), twiddles
// per lane, and the place of its lanes' twiddles in the table
constexpr int FFT_REG_MIN = 6, FFT_REG_MAX = 12;
constexpr int fft_reg_p8(int logl) { return logl / 3; }
constexpr int fft_reg_last(int logl) { return 1 << (logl % 3); }
constexpr int fft_reg_ntw(int logl) {
    const int last = fft_reg_last(logl);
    return 7 * (fft_reg_p8(logl) - 1) + (last == 1 ? 0 : (last - 1) * (8 / last));
}
constexpr int fft_reg_at(int logl) {
    int n = 0;
    for (int l = FFT_REG_MIN; l < logl; ++l) n += fft_reg_ntw(l) << (l - 3);
    return n;
}
static __device__ float2 g_fft_lane32[fft_reg_at(FFT_REG_MAX + 1)];
static __device__ double2 g_fft_lane64[fft_reg_at(FFT_REG_MAX + 1)];

// Numerator j of twiddle n of lane t, W = e^{-2 pi i j / L}.
__host__ __device__ inline int fft_reg_angle(int logl, int n, int t) {
    const int p = n / 7 + 1;  // pass
    if (p < fft_reg_p8(logl)) {
        const int ns = 1 << (3 * p);
        return (t % ns) * (n % 7 + 1) * ((1 << logl) / (8 * ns));
    }
    const int r = fft_reg_last(logl), e = n - 7 * (fft_reg_p8(logl) - 1);
    const int s = e / (r - 1), m = e % (r - 1) + 1;
    return (t + (1 << (logl - 3)) * s) * m;
}

template <typename R>
struct FT;
template <>
struct FT<float> {
    typedef float2 C;
    __device__ static C tw(int j) { return g_fft_tw32[j]; }
    __device__ static C lane(int i) { return g_fft_lane32[i]; }
    __device__ static C mk(float a, float b) { return make_float2(a, b); }
    // W_L^m for arbitrary L (four-step twiddles), evaluated in double
    __device__ static C wl(long long m, long long L, bool inv) {
        double s, c;
        sincospi((inv ? 2.0 : -2.0) * (double)m / (double)L, &s, &c);
        return make_float2((float)c, (float)s);
    }
};
template <>
struct FT<double> {
    typedef double2 C;
    __device__ static C tw(int j) { return g_fft_tw64[j]; }
    __device__ static C lane(int i) { return g_fft_lane64[i]; }
    __device__ static C mk(double a, double b) { return make_double2(a, b); }
    __device__ static C wl(long long m, long long L, bool inv) {
        double s, c;
        sincospi((inv ? 2.0 : -2.0) * (double)m / (double)L, &s, &c);
        return make_double2(c, s);
    }
};

template <typename C>
__device__ __forceinline__ C cmul2(C a, C b) {
    C r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
// a * b, or a * conj(b) for the inverse transform
template <bool INV, typename C>
__device__ __forceinline__ C cmul_tw(C a, C b) {
    C r;
    if constexpr (INV) {
        r.x = a.x * b.x + a.y * b.y;
        r.y = a.y * b.x - a.x * b.y;
    } else {
        r.x = a.x * b.x - a.y * b.y;
        r.y = a.x * b.y + a.y * b.x;
    }
    return r;
}
template <typename C>
__device__ __forceinline__ C cadd2(C a, C b) {
    C r;
    r.x = a.x + b.x;
    r.y = a.y + b.y;
    return r;
}
template <typename C>
__device__ __forceinline__ C csub2(C a, C b) {
    C r;
    r.x = a.x - b.x;
    r.y = a.y - b.y;
    return r;
}
// a * -i (forward) or a * i (inverse)
template <bool INV, typename C>
__device__ __forceinline__ C crot(C a) {
    C r;
    r.x = INV ? -a.y : a.y;
    r.y = INV ? a.x : -a.x;
    return r;
}

template <bool INV, typename C>
__device__ __forceinline__ void dft2(C &a, C &b) {
    const C t = a;
    a = cadd2(t, b);
    b = csub2(t, b);
}
template <bool INV, typename C>
__device__ __forceinline__ void dft4(C &a, C &b, C &c, C &d) {
    const C s0 = cadd2(a, c), d0 = csub2(a, c), s1 = cadd2(b, d), d1 = crot<INV>(csub2(b, d));
    a = cadd2(s0, s1);
    b = cadd2(d0, d1);
    c = csub2(s0, s1);
    d = csub2(d0, d1);
}
template <bool INV, typename R, typename C>
__device__ __forceinline__ void dft8(C (&v)[8]) {
    const R h = (R)0.70710678118654752440;
    C e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    C o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4<INV>(e0, e1, e2, e3);
    dft4<INV>(o0, o1, o2, o3);
    // o_k * W_8^k
    C w1 = crot<INV>(o1), w3 = crot<INV>(o3);
    w1 = cadd2(o1, w1);  // (1 -+ i) o1
    w3 = csub2(w3, o3);  // (-1 -+ i) o3
    w1.x *= h;
    w1.y *= h;
    w3.x *= h;
    w3.y *= h;
    const C w2 = crot<INV>(o2);
    v[0] = cadd2(e0, o0);
    v[1] = cadd2(e1, w1);
    v[2] = cadd2(e2, w2);
    v[3] = cadd2(e3, w3);
    v[4] = csub2(e0, o0);
    v[5] = csub2(e1, w1);
    v[6] = csub2(e2, w2);
    v[7] = csub2(e3, w3);
}

template <typename R, int LOGL>
struct RegFft {
    using C = typename FT<R>::C;
    static constexpr int L = 1 << LOGL;
    static constexpr int NT = L / 8;                      // lanes per transform
    static constexpr int P8 = fft_reg_p8(LOGL);
    static constexpr int LAST = fft_reg_last(LOGL);
    static constexpr int NTW = fft_reg_ntw(LOGL);
    static constexpr int THREADS = NT < 256 ? 256 : NT;   // workgroup
    static constexpr int TPW = THREADS / NT;              // transforms per workgroup
    static constexpr int PITCH = L + L / 8;               // LDS values per transform
    __device__ static constexpr int at(int i) { return i + (i >> 3); }

    C tw[NTW];

    // the lane's twiddles for every pass after the first
    __device__ __forceinline__ void init(int t) {
#pragma unroll
        for (int n = 0; n < NTW; ++n) tw[n] = FT<R>::lane(fft_reg_at(LOGL) + n * NT + t);
    }

    // lane t's points t + NT * j are row(t) + j * ROW in LDS
    static constexpr int ROW = NT + NT / 8;
    __device__ __forceinline__ static int row(int t) { return t + (t >> 3); }

    // writes pass output (index q of radix-8 butterflies, NS = product of the
    // earlier radices) and reads the lane's points of the next pass
    template <int NS>
    __device__ __forceinline__ static void exchange(C (&v)[8], C *lds, int t) {
        // point (t / NS) * 8 NS + t % NS + m * NS
        C *w = lds + (NS == 1 ? 9 * t : at(t / NS * NS * 8 + t % NS));
        const C *r = lds + row(t);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 8; ++m) w[NS == 1 ? m : m * (NS + NS / 8)] = v[m];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = r[j * ROW];
    }

    template <bool INV, int NS>
    __device__ __forceinline__ void pass8(C (&v)[8], C *lds, int t) const {
        constexpr int first = NS == 8 ? 0 : NS == 64 ? 7 : 14;
        exchange<NS / 8>(v, lds, t);
#pragma unroll
        for (int m = 1; m < 8; ++m) v[m] = cmul_tw<INV>(v[m], tw[first + m - 1]);
        dft8<INV, R>(v);
    }

    // In place over the workgroup's transforms; every lane of the workgroup
    // takes part. lds: this transform's PITCH values.
    template <bool INV>
    __device__ __forceinline__ void run(C (&v)[8], C *lds, int t) const {
        dft8<INV, R>(v);
        if constexpr (P8 > 1) pass8<INV, 8>(v, lds, t);
        if constexpr (P8 > 2) pass8<INV, 64>(v, lds, t);
        if constexpr (P8 > 3) pass8<INV, 512>(v, lds, t);
        if constexpr (LAST > 1) {
            int n = 7 * (P8 - 1);
            exchange<(1 << (3 * (P8 - 1)))>(v, lds, t);
#pragma unroll
            for (int s = 0; s < 8 / LAST; ++s) {
                // butterfly t + NT * s: points t + NT * (s + m * 8 / LAST)
                if constexpr (LAST == 2) {
                    v[s + 4] = cmul_tw<INV>(v[s + 4], tw[n++]);
                    dft2<INV>(v[s], v[s + 4]);
                } else {
#pragma unroll
                    for (int m = 1; m < 4; ++m) v[s + 2 * m] = cmul_tw<INV>(v[s + 2 * m], tw[n++]);
                    dft4<INV>(v[s], v[s + 2], v[s + 4], v[s + 6]);
                }
            }
        }
    }
};

}  // namespace afhip
