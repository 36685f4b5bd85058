// The af_convolve* C API of libafhip and its backend host layer.
//
// Dispatch restates src/api/c/convolve.cpp (rank fallback, domain heuristic,
// batch-kind detection, dtype -> accumulator map, asserts and error codes).
// The backend layer ("detail", src/backend/cpu/convolve.cpp:38-243) computes
// output dims, allocates from the stream-ordered pool and queues the gfx950
// kernels through the kernel C ABI (include/afhip_kernels.h).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <memory>
#include <vector>
#include <string>
#include <functional>

#include "../../include/af/array.h"
#include "../../include/af/ml.h"
#include "../../include/af/signal.h"
#include "../../include/afhip_kernels.h"
#include "autotune.hpp"
#include "nn_wgemm.hpp"
#include "nn_x3.hpp"
#include "runtime.hpp"

namespace afhip {

// AF_BATCH_KIND, src/backend/common/internal_enums.hpp:15-22
enum BatchKind {
    BATCH_NONE = 1,
    BATCH_LHS = 2,
    BATCH_RHS = 3,
    BATCH_SAME = 4,
    BATCH_DIFF = 5,
    BATCH_UNSUPPORTED = 6
};

// src/api/c/convolve.cpp:77-97
static BatchKind identify_batch_kind(int rank, const dim4 &s, const dim4 &f) {
    const dim_t sn = s.ndims(), fn = f.ndims();
    if (sn == rank && fn == rank) return BATCH_NONE;
    if (sn == rank && (fn > rank && fn <= AF_MAX_DIMS)) return BATCH_RHS;
    if ((sn > rank && sn <= AF_MAX_DIMS) && fn == rank) return BATCH_LHS;
    if ((sn > rank && sn <= AF_MAX_DIMS) && (fn > rank && fn <= AF_MAX_DIMS)) {
        bool match = true, inter = true;
        for (int i = rank; i < AF_MAX_DIMS; ++i) {
            match &= s[i] == f[i];
            inter &= (s[i] == 1 || f[i] == 1 || s[i] == f[i]);
        }
        if (match) return BATCH_SAME;
        return inter ? BATCH_DIFF : BATCH_UNSUPPORTED;
    }
    return BATCH_UNSUPPORTED;
}

// src/api/c/convolve.cpp:99-130
static bool is_freq_domain(int rank, const dim4 &s, const dim4 &f, af_conv_domain domain) {
    if (domain == AF_CONV_FREQ) return true;
    if (domain != AF_CONV_AUTO) return false;
    if (identify_batch_kind(rank, s, f) == BATCH_DIFF) return true;
    dim_t kbatch = 1;
    for (int i = 3; i >= rank; --i) kbatch *= f[i];
    if (kbatch >= 10) return true;
    if (rank == 1 && f[0] > 128) return true;
    if (rank == 2) {
        if (f[0] > 17 || f[1] > 17) return true;
        if (f[0] != f[1] && f[0] > 5) return true;
    }
    if (rank == 3 && (f[0] > 5 || f[1] > 5 || f[2] > 5)) return true;
    return false;
}

// Accumulator dtype per signal dtype: src/api/c/convolve.cpp:155-209.
static af_dtype acc_type(af_dtype t) {
    switch ((int)t) {
        case c32: return c32;
        case c64: return c64;
        case f32: return f32;
        case f64: return f64;
        case u32:
        case s32:
        case u16:
        case s16:
        case u64:
        case s64:
        case u8:
        case s8:
        case b8: return f32;
        default: TYPE_ERROR(1, t);
    }
}

// castArray<accT>: a device copy converted to accT (shares storage when the
// type already matches).
static std::shared_ptr<Buffer> cast_buffer(const ArrayImpl &a, af_dtype to) {
    if (a.type == to) return a.buf;
    const dim_t n = a.elements();
    auto b = scratch((size_t)n * dtype_size(to));
    check_k(afhip_k_cast(to, b->ptr, a.type, a.data(), n, stream()), "cast");
    return b;
}

// ---------------------------------------------------------------- detail
namespace detail {

// Output dims: src/backend/cpu/convolve.cpp:44-58
static dim4 conv_out_dims(const dim4 &s, const dim4 &f, BatchKind kind, int rank, bool expand) {
    dim4 o(1, 1, 1, 1);
    if (expand) {
        for (int d = 0; d < AF_MAX_DIMS; ++d) {
            if (kind == BATCH_NONE || kind == BATCH_RHS)
                o[d] = s[d] + f[d] - 1;
            else
                o[d] = d < rank ? s[d] + f[d] - 1 : s[d];
        }
    } else {
        o = s;
        if (kind == BATCH_RHS)
            for (int i = rank; i < AF_MAX_DIMS; ++i) o[i] = f[i];
    }
    return o;
}

// cpu::convolve<T, accT>, src/backend/cpu/convolve.cpp:38-66
static af_array convolve(const ArrayImpl &sig, const ArrayImpl &filt, BatchKind kind, int rank,
                         bool expand) {
    const af_dtype at = acc_type(sig.type);
    auto fbuf = cast_buffer(filt, at);
    const dim4 od = conv_out_dims(sig.dims, filt.dims, kind, rank, expand);
    NewHandle out(make_handle(sig.type, od));
    if (od.elements() > 0) {
        check_k(afhip_k_convolve(sig.type, out.data(), od.d, sig.data(), sig.dims.d, fbuf->ptr,
                                 filt.dims.d, (int)kind, rank, expand ? 1 : 0, stream()),
                "convolve");
    }
    return out.release();
}

// cpu::convolve2<T, accT> (separable), src/backend/cpu/convolve.cpp:68-99
static af_array convolve2_sep(const ArrayImpl &sig, const std::shared_ptr<Buffer> &cf, dim_t cflen,
                              const std::shared_ptr<Buffer> &rf, dim_t rflen, bool expand) {
    dim4 od = sig.dims;
    dim4 td = sig.dims;
    if (expand) {
        od[0] += cflen - 1;
        od[1] += rflen - 1;
        td[0] += cflen - 1;
    }
    NewHandle out(make_handle(sig.type, od));
    if (od.elements() == 0) return out.release();
    // FP32 with filters of up to AFHIP_SEP_FUSED_MAX_TAPS runs fused (the
    // intermediate never leaves the chip); everything else runs the two
    // passes through the reference's T-typed temp.
    std::shared_ptr<Buffer> tmp;
    const bool fused = sig.type == f32 && cflen <= AFHIP_SEP_FUSED_MAX_TAPS &&
                       rflen <= AFHIP_SEP_FUSED_MAX_TAPS;
    if (!fused) tmp = scratch((size_t)td.elements() * dtype_size(sig.type));
    check_k(afhip_k_convolve2_sep(sig.type, out.data(), od.d, sig.data(), sig.dims.d, cf->ptr,
                                  cflen, rf->ptr, rflen, expand ? 1 : 0, tmp ? tmp->ptr : nullptr,
                                  stream()),
            "convolve2_sep");
    return out.release();
}

// convolve2_unwrap output size, src/backend/cpu/convolve.cpp:130-135
// (C++ integer division truncates toward zero).
static dim_t nn_out(dim_t s, dim_t f, dim_t st, dim_t pd, dim_t dl) {
    return 1 + (s + 2 * pd - (((f - 1) * dl) + 1)) / st;
}

struct NNGeom {
    dim4 x, w, y;
    long long st[2], pd[2], dl[2];
};

static NNGeom nn_geom(const dim4 &x, const dim4 &w, const dim4 &stride, const dim4 &padding,
                      const dim4 &dilation) {
    NNGeom g;
    g.x = x;
    g.w = w;
    for (int i = 0; i < 2; ++i) {
        g.st[i] = stride[i];
        g.pd[i] = padding[i];
        g.dl[i] = dilation[i];
    }
    const dim_t ow = nn_out(x[0], w[0], stride[0], padding[0], dilation[0]);
    const dim_t oh = nn_out(x[1], w[1], stride[1], padding[1], dilation[1]);
    g.y = dim4(ow, oh, w[3], x[3]);
    return g;
}

static void check_nn_geom(const NNGeom &g) {
    // The kernels index with 32-bit extents and need positive sizes.
    for (int i = 0; i < 4; ++i) {
        DIM_ASSERT(1, g.x[i] >= 0 && g.x[i] < (1LL << 31));
        DIM_ASSERT(2, g.w[i] >= 0 && g.w[i] < (1LL << 31));
    }
    DIM_ASSERT(1, g.y[0] >= 0 && g.y[1] >= 0);
    ARG_ASSERT(3, g.st[0] > 0 && g.st[1] > 0);
    ARG_ASSERT(7, g.dl[0] > 0 && g.dl[1] > 0);
}

// f64 inputs run the direct FP64 kernels (afhip_k_conv2_nn_f64); the MFMA
// implicit-GEMM kernels take FP32 and 16-bit operands only.

// The patch-staged kernels serve the forward pass and the stride-1 data
// gradient when the input patch fits in LDS, the row-staged kernel the filter
// gradient of 16-bit operands; AFHIP_NN_GATHER=1 forces the gather kernels
// (the tests use it to cover both paths).
static int device_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        return 256;
    return n;
}

// ---- NN variant choice. Layers that fill the chip with the patch kernels'
// tiles, strided data gradients that fill it phase by phase and all filter
// gradients go by rules on the sizes (patch_by_rule, rows_by_rule): no timing on
// the first call, and the same kernel, so the same bits, on every run. The other
// forward passes and data gradients are the autotuner's (autotune.cpp): it times
// the candidate variants (the patch kernels where they serve; the GEMM with
// splits of the reduction) on the first call of a geometry and caches the
// fastest under a key of (pass, dtypes, precision, dims, stride, padding,
// dilation). Under stream capture only cached choices are used.
// AFHIP_NN_AUTOTUNE=0 (or an explicit AFHIP_NN_SPLIT) keeps built-in rules there
// too.
static bool nn_autotune_on() {
    const char *a = std::getenv("AFHIP_NN_AUTOTUNE");
    const char *sp = std::getenv("AFHIP_NN_SPLIT");
    return !(a && a[0] == '0') && !(sp && sp[0] >= '1' && sp[0] <= '9');
}

static bool stream_capturing() {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream(), &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// The key names the arithmetic (the MMA operand mode), not the storage
// types, so that calls computing the same products (f32 arrays at BF16
// precision and bf16 arrays; f32 and 16-bit outputs) run the same variant and
// give the same sums.
static std::string nn_key(const char *tag, int pass, const ArrayImpl &in, af_dtype, int precision,
                          const NNGeom &g) {
    const int mode = precision != AFHIP_PRECISION_DEFAULT ? precision
                     : in.type == f32                     ? (int)AFHIP_PRECISION_F32
                     : in.type == afhip_bf16              ? (int)AFHIP_PRECISION_BF16
                                                          : (int)AFHIP_PRECISION_F16;
    // the storage type too: f32 arrays at a 16-bit precision run other
    // kernels (element gather) than 16-bit arrays (channel-last copies)
    std::string k = std::string(tag) + ":p" + std::to_string(pass) + ":m" + std::to_string(mode) + ":t" +
                    std::to_string((int)in.type);
    for (int i = 0; i < 4; ++i) k += (i ? "," : ":x") + std::to_string(g.x[i]);
    for (int i = 0; i < 4; ++i) k += (i ? "," : ":w") + std::to_string(g.w[i]);
    k += ":s" + std::to_string(g.st[0]) + "," + std::to_string(g.st[1]) + ":pd" + std::to_string(g.pd[0]) + "," +
         std::to_string(g.pd[1]) + ":d" + std::to_string(g.dl[0]) + "," + std::to_string(g.dl[1]);
    return k;
}

struct NNCand {
    const char *name;
    int split;
    std::function<void()> run;
};

// Index of the variant to run: the autotuner's (timing them now if the key
// is new), or -1 for the built-in rule. The list depends on more than the
// layer (switches in the environment, the result's type, the device's CUs), so
// its names are part of the key: an index is only ever read back for the list
// it was chosen from.
static int nn_pick(std::string key, const std::vector<NNCand> &cands) {
    if (cands.size() < 2 || !nn_autotune_on()) return -1;
    for (size_t i = 0; i < cands.size(); ++i)
        key += (i ? "," : ":of ") + std::string(cands[i].name) + std::to_string(cands[i].split);
    if (stream_capturing()) {
        const int r = autotune_lookup(key);
        return r >= 0 && r < (int)cands.size() ? r : -1;
    }
    return autotune_pick(key, (int)cands.size(), [&](int c) { cands[c].run(); });
}

static const int kSplitCands[] = {1, 2, 4, 8, 16};

static void run_gemm_split(int pass, const ArrayImpl &in, const ArrayImpl &w, af_dtype out_type, int precision,
                           void *out, const NNGeom &g, int nsplit) {
    const long long need = afhip_k_conv2_nn_gemm_split_workspace(pass, in.type, precision, g.x.d, g.w.d, g.y.d,
                                                                 g.st, g.pd, g.dl, nsplit);
    std::shared_ptr<Buffer> ws;
    if (need > 0) ws = scratch((size_t)need);
    check_k(afhip_k_conv2_nn_gemm_split(pass, in.type, out_type, precision, out, in.data(), w.data(), g.x.d,
                                        g.w.d, g.y.d, g.st, g.pd, g.dl, nsplit, ws ? ws->ptr : nullptr, need,
                                        stream()),
            pass == 0 ? "convolve2_nn" : "convolve2_gradient_nn");
}

// FP32 on the BF16 matrix cores in three parts per operand: f32 arrays and
// results at their own precision. AFHIP_NN_X3=0 leaves it out, =1 takes it wherever it
// serves.
static int x3_env() {
    const char *e = std::getenv("AFHIP_NN_X3");
    return e && (e[0] == '0' || e[0] == '1') ? e[0] - '0' : -1;
}
static bool x3_serves(int pass, const ArrayImpl &in, af_dtype out_type, int precision, const NNGeom &g) {
    if (in.type != f32 || out_type != f32 || (precision != AFHIP_PRECISION_DEFAULT && precision != AFHIP_PRECISION_F32)) return false;
    const char *gather = std::getenv("AFHIP_NN_GATHER");
    if (x3_env() == 0 || (gather && gather[0] == '1')) return false;
    return nn_x3_workspace(pass, g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, 1) > 0;
}
static void run_x3(int pass, const ArrayImpl &in, const ArrayImpl &w, void *out, const NNGeom &g, int nsplit) {
    const long long need = nn_x3_workspace(pass, g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, nsplit);
    auto ws = scratch((size_t)need);
    check_k(nn_x3(pass, out, in.data(), w.data(), g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, nsplit, ws->ptr, need,
                  stream()),
            pass == 0 ? "convolve2_nn" : "convolve2_gradient_nn");
}

static void run_patch_kernels(int pass, const ArrayImpl &in, const ArrayImpl &w, af_dtype out_type, int precision,
                              void *out, const NNGeom &g, long long need) {
    auto ws = scratch((size_t)need);
    check_k(afhip_k_conv2_nn_patch(pass, in.type, out_type, precision, out, in.data(), w.data(), g.x.d, g.w.d,
                                   g.y.d, g.st, g.pd, g.dl, ws->ptr, need, stream()),
            pass == 0 ? "convolve2_nn" : "convolve2_gradient_nn");
}

// Candidates: the patch kernels, where they serve, then the GEMM with the split
// counts worth a try. Splitting pays only where the GEMM's own tiles leave CUs
// idle.
static std::vector<NNCand> nn_candidates(int pass, const ArrayImpl &in, const ArrayImpl &w, af_dtype out_type,
                                         int precision, void *out, const NNGeom &g,
                                         std::function<void()> patch) {
    std::vector<NNCand> c;
    if (patch) c.push_back({"patch/", 1, std::move(patch)});
    const dim4 &o = pass == 0 ? g.y : g.x;
    const long long tiles = (o[2] + 127) / 128 * ((o[0] * o[1] * o[3] + 127) / 128);
    if (x3_serves(pass, in, out_type, precision, g))
        for (int sp : {1, 2, 4})
            if (sp == 1 || tiles < device_cus())
                c.push_back({"x3/", sp, [=, &in, &w, &g] { run_x3(pass, in, w, out, g, sp); }});
    for (int sp : kSplitCands)
        if (sp == 1 || tiles < device_cus())
            c.push_back({"gemm/", sp, [=, &in, &w, &g] { run_gemm_split(pass, in, w, out_type, precision, out, g, sp); }});
    return c;
}

// first, or second where the device has no room for first's workspace: copies
// of both operands, up to 2 GiB each, where the kernels that do without need
// the packed weights or nothing. Workspaces are allocated before any launch.
template <typename A, typename B>
static void or_with_less_memory(A &&first, B &&second) {
    try {
        first();
    } catch (const AfError &e) {
        if (e.code() != AF_ERR_NO_MEM) throw;
        second();
    }
}

// Whether the GEMM reads channel-last copies (operands at their own precision,
// copies within its offsets) rather than single elements.
static bool gemm_copies(int pass, const ArrayImpl &in, int precision, const NNGeom &g) {
    return afhip_k_conv2_nn_gemm_split_workspace(pass, in.type, precision, g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, 1) > 0;
}

// Whether the rows of x and y are whole vectors of 16 bytes.
static bool whole_rows(const NNGeom &g, af_dtype t) {
    const dim_t v = t == f32 ? 4 : 8;
    return g.x[0] % v == 0 && g.y[0] % v == 0;
}

// Of the layers whose patch tiles fill the chip, those that the patch kernels
// run faster than the GEMM (x3 for f32), us:
//  * f32: 9 to 16 reduction channels, one chunk of the patch kernels and half of
//    a GEMM slice (60x60x16x32 -> 16, 3x3: 31 and 43), and 1x1 filters that do
//    not widen the channels, where the copies cost as much as the product
//    (64x64x128x32 -> 128: 63 and 74; to 256 from 56x56x64x32: 73 and 58). Else
//    the GEMM (28x28x128x64 -> 128, 3x3: 171 and 121; 62x62x128x16 -> 128: 189
//    and 145);
//  * 16-bit: few channels (57x57x3x64 -> 64, 3x3: 37 and 44; to more than 32
//    over odd rows, or with more taps, the GEMM, 68x35x16x27 -> 128: 27 and 22;
//    54x78x16x22 -> 16, 5x5, step: 127 and 101), and many whole rows
//    under the weights-resident kernel or under pipelined stages that do not
//    widen the channels (56x56x64x32 -> 128, 3x3: 29 and 39; 64x64x128x32 ->
//    128, 1x1: 29 and 32; 32x32x96x64 -> 96, 5x5: 57 and 64). Else the GEMM
//    (28x28x128x64 -> 128: 77 and 37; 48x48x64x64 -> 32, 5x5: 83 and 71;
//    96x96x64x32 -> 64, 5x5, stride 2: 178 and 53; rows of 8 pixels 269 and
//    110; 16x16x128x16 -> 96: 16.8 and 14.0).
static bool patch_by_rule(int pass, const ArrayImpl &in, const NNGeom &g) {
    const dim_t R = pass == 0 ? g.x[2] : g.w[3], M = pass == 0 ? g.w[3] : g.x[2], taps = g.w[0] * g.w[1];
    const bool whole = whole_rows(g, in.type), unit = g.st[0] == 1 && g.st[1] == 1;
    if (in.type == f32) return whole && ((R > 8 && R <= 16) || (taps == 1 && R >= M));
    if (taps <= 9 && (R <= 8 || (R <= 16 && (whole || M <= 32)))) return true;
    if (!whole || g.x[0] < 16 || g.y[0] * g.y[1] * g.y[3] < 16384) return false;
    if (taps == 1) return unit && R >= M;
    return taps <= 9 ? unit || taps == 9 : unit && R >= 96;
}

// AFHIP_NN_SMALL=0 keeps every served layer on the patch kernels. Built-in rule
// for the autotuned layers: the patch kernels when they launch at least a
// quarter of the CUs' workgroups.
static bool run_patch(int pass, const ArrayImpl &in, const ArrayImpl &w, af_dtype out_type,
                      int precision, void *out, const NNGeom &g) {
    const char *env = std::getenv("AFHIP_NN_GATHER");
    if (env && env[0] == '1') return false;
    const long long need = afhip_k_conv2_nn_patch_workspace(pass, in.type, precision, g.x.d, g.w.d,
                                                            g.y.d, g.st, g.pd, g.dl);
    if (need <= 0) return false;
    const bool x3 = x3_serves(pass, in, out_type, precision, g);
    if (x3_env() == 1 && x3) {
        run_x3(pass, in, w, out, g, 1);
        return true;
    }
    auto patch = [=, &in, &w, &g] { run_patch_kernels(pass, in, w, out_type, precision, out, g, need); };
    const char *sm = std::getenv("AFHIP_NN_SMALL");
    if (sm && sm[0] == '0') {
        patch();
        return true;
    }
    const long long tiles = afhip_k_conv2_nn_patch_tiles(pass, in.type, precision, g.x.d, g.w.d, g.y.d, g.st, g.pd,
                                                         g.dl);
    if (tiles >= device_cus()) {
        const bool gemm = in.type == f32 ? x3 : gemm_copies(pass, in, precision, g);
        if (!gemm || patch_by_rule(pass, in, g))
            patch();
        else if (x3)
            or_with_less_memory([&] { run_x3(pass, in, w, out, g, 1); }, patch);
        else
            or_with_less_memory([&] { run_gemm_split(pass, in, w, out_type, precision, out, g, 1); }, patch);
        return true;
    }
    const auto cands = nn_candidates(pass, in, w, out_type, precision, out, g, patch);
    int c = nn_pick(nn_key("nn3", pass, in, out_type, precision, g), cands);
    if (c < 0) c = tiles * 4 >= device_cus() ? 0 : -1;
    if (c >= 0)
        or_with_less_memory(cands[c].run, patch);
    else
        run_gemm_split(pass, in, w, out_type, precision, out, g, 0);
    return true;
}

// The GEMM for every other geometry, its split count autotuned (built-in
// rule: split when that fills the chip).
static void run_gemm(int pass, const ArrayImpl &in, const ArrayImpl &w, af_dtype out_type, int precision,
                     void *out, const NNGeom &g) {
    if (x3_env() == 1 && x3_serves(pass, in, out_type, precision, g)) {
        run_x3(pass, in, w, out, g, 1);
        return;
    }
    const auto cands = nn_candidates(pass, in, w, out_type, precision, out, g, nullptr);
    const int c = nn_pick(nn_key("nn_gemm3", pass, in, out_type, precision, g), cands);
    if (c >= 0)
        or_with_less_memory(cands[c].run, [&] { run_gemm_split(pass, in, w, out_type, precision, out, g, 1); });
    else
        run_gemm_split(pass, in, w, out_type, precision, out, g, 0);
}

static af_dtype nn_out_type(af_dtype in, af_dtype requested) {
    if ((int)requested == -1) return in;
    return requested;
}

// Refuses the combinations of storage, arithmetic and result that the kernels
// refuse, where no kernel runs.
static void check_nn_types(af_dtype in, af_dtype out, int precision) {
    ARG_ASSERT(9, precision >= AFHIP_PRECISION_DEFAULT && precision <= AFHIP_PRECISION_F32);
    const int own = in == afhip_bf16 ? AFHIP_PRECISION_BF16 : AFHIP_PRECISION_F16;
    if (in != f32 && in != f64 && precision != AFHIP_PRECISION_DEFAULT && precision != own) TYPE_ERROR(1, in);
    if (out != in && (out != f32 || in == f64)) TYPE_ERROR(10, out);
}

// cpu::convolve2<T> (NN forward), src/backend/cpu/convolve.cpp:160-167
static af_array conv2_nn(const ArrayImpl &x, const ArrayImpl &w, const NNGeom &g, int precision,
                         af_dtype out_type) {
    NewHandle out(make_handle(out_type, g.y));
    if (g.y.elements() == 0) return out.release();
    // outputs of padding alone: the kernels read at least one pixel and one tap
    if (g.x.elements() == 0 || g.w.elements() == 0) {
        check_nn_types(x.type, out_type, precision);
        check_k(afhip_k_fill(out_type, out.data(), 0.0, g.y.elements(), stream()), "fill");
        return out.release();
    }
    if (x.type == f64) {
        check_k(afhip_k_conv2_nn_f64(0, out.data(), x.data(), w.data(), g.x.d, g.w.d, g.y.d, g.st,
                                     g.pd, g.dl, stream()),
                "convolve2_nn");
        return out.release();
    }
    if (run_patch(0, x, w, out_type, precision, out.data(), g)) return out.release();
    run_gemm(0, x, w, out_type, precision, out.data(), g);
    return out.release();
}

// cpu::conv2DataGradient<T>, src/backend/cpu/convolve.cpp:179-211
static af_array conv2_data_grad(const ArrayImpl &dy, const ArrayImpl &x, const ArrayImpl &w,
                                const NNGeom &g, int precision, af_dtype out_type) {
    NewHandle out(make_handle(out_type, g.x));
    if (g.x.elements() == 0) return out.release();
    void *o = out.data();
    if (dy.elements() == 0 || g.w.elements() == 0) {
        check_k(afhip_k_fill(out_type, o, 0.0, g.x.elements(), stream()), "fill");
        return out.release();
    }
    if (x.type == f64) {
        check_k(afhip_k_conv2_nn_f64(1, o, dy.data(), w.data(), g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl,
                                     stream()),
                "convolve2_gradient_nn");
        return out.release();
    }
    if (run_patch(1, dy, w, out_type, precision, o, g)) return out.release();
    // Strided layers whose phases fill the chip: the GEMM over phase-ordered
    // pixels where it reads channel-last copies (57x57x64x64 -> 128, 3x3, stride
    // 2: BF16 58 us, FP32 104 us; 302 and 349 us as polyphase stride-1
    // convolutions on the patch kernels, which need a launch per phase to pack,
    // convolve and scatter), the polyphase split elsewhere. AFHIP_NN_POLY=1 takes
    // the split, AFHIP_NN_GATHER=1 leaves it out.
    const char *gather = std::getenv("AFHIP_NN_GATHER"), *pe = std::getenv("AFHIP_NN_POLY");
    const long long pb = gather && gather[0] == '1'
                             ? 0
                             : afhip_k_conv2_nn_dgrad_poly_workspace(x.type, out_type, precision, g.x.d, g.w.d, g.y.d,
                                                                     g.st, g.pd, g.dl);
    if (pb > 0) {
        const auto poly = [&] {
            auto ws = scratch((size_t)pb);
            check_k(afhip_k_conv2_nn_dgrad_poly(x.type, out_type, precision, o, dy.data(), w.data(), g.x.d, g.w.d,
                                                g.y.d, g.st, g.pd, g.dl, ws->ptr, pb, stream()),
                    "convolve2_gradient_nn");
        };
        const bool gemm = !(pe && pe[0] == '1');
        if (gemm && x3_serves(1, dy, out_type, precision, g))
            or_with_less_memory([&] { run_x3(1, dy, w, o, g, 1); }, poly);
        else if (gemm && gemm_copies(1, dy, precision, g))
            or_with_less_memory([&] { run_gemm_split(1, dy, w, out_type, precision, o, g, 1); }, poly);
        else
            poly();
        return out.release();
    }
    run_gemm(1, dy, w, out_type, precision, o, g);
    return out.release();
}

// The row-staged kernels where they serve (filter sides 1 and 3), else the
// element gather.
static void wgrad_rows_or_gather(const ArrayImpl &dy, const ArrayImpl &x, const NNGeom &g, int precision,
                                 af_dtype out_type, void *o, bool gather) {
    const long long rb = gather ? 0
                                : afhip_k_conv2_nn_wgrad_rows_workspace(x.type, precision, g.x.d, g.w.d, g.y.d, g.st,
                                                                        g.pd, g.dl);
    if (rb > 0) {
        auto ws = scratch((size_t)rb);
        check_k(afhip_k_conv2_nn_wgrad_rows(x.type, out_type, precision, o, x.data(), dy.data(), g.x.d, g.w.d, g.y.d,
                                            g.st, g.pd, g.dl, ws->ptr, rb, stream()),
                "convolve2_gradient_nn");
        return;
    }
    const long long wsb = afhip_k_conv2_nn_wgrad_workspace(g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl);
    std::shared_ptr<Buffer> ws;
    if (wsb > 0) ws = scratch((size_t)wsb);
    check_k(afhip_k_conv2_nn_wgrad(x.type, out_type, precision, o, x.data(), dy.data(), g.x.d, g.w.d, g.y.d, g.st,
                                   g.pd, g.dl, ws ? ws->ptr : nullptr, wsb, stream()),
            "convolve2_gradient_nn");
}

// Of the filter gradients that the row-staged kernels serve, those that they run
// faster than the GEMM over channel-last copies, us: many whole rows, and
//  * f32: 1x1 filters of one tile (56x56x64x32 -> 64: 41 and 45; 112x112x64x8 ->
//    64: 38 and 45). Else the GEMM (56x56x64x32 -> 128, 3x3: 205 and 124;
//    41x67x16x30 -> 16, 1x1: 50 and 32);
//  * 16-bit: rows that fill four fifths of the kernels' 32-pixel steps, with
//    a full tile of filters or channels and a quarter of one of the other, and
//    1x1 filters of few tiles (56x56x64x32 -> 128, 3x3: 42 and 49; 64x64x64x64
//    -> 64: 46 and 64; 32x32x256x32 -> 64, 1x1: 19 and 25). Else the GEMM
//    (40x40x64x32 -> 64: 34 and 27; 56x56x16x32 -> 16: 36 and 29; 72x72x3x32 ->
//    64: 53 and 46; 28x28x128x32 -> 128: 72 and 33; 72x70x48x3 -> 256: 35 and
//    28; 32x66x32x22 -> 64: 30 and 23; 80x80x256x4 -> 256, 1x1: 42 and 29).
static bool rows_by_rule(const ArrayImpl &x, const NNGeom &g) {
    if (!whole_rows(g, x.type)) return false;
    const dim_t lo = std::min(g.x[2], g.w[3]), hi = std::max(g.x[2], g.w[3]), px = g.y[0] * g.y[1] * g.y[3];
    const dim_t taps = g.w[0] * g.w[1], ow = g.y[0];
    if (x.type == f32) return taps == 1 && hi <= 64 && px >= 65536;
    return px >= 32768 && hi >= 64 && lo >= 16 && lo * hi * px >= 200000000 && ow >= 32 && ow * 5 >= (ow + 31) / 32 * 32 * 4 &&
           (taps > 1 || lo * hi * g.st[0] * g.st[1] <= 16384);
}

// By that rule, for any other geometry the GEMM. AFHIP_NN_WG=0 leaves the GEMM
// out, =1 takes it wherever it serves.
static void run_wgrad(const ArrayImpl &dy, const ArrayImpl &x, const NNGeom &g, int precision, af_dtype out_type,
                      void *o) {
    const char *env = std::getenv("AFHIP_NN_GATHER"), *wg = std::getenv("AFHIP_NN_WG");
    const bool gather = env && env[0] == '1';
    const bool own = precision == AFHIP_PRECISION_DEFAULT ||
                     precision == (x.type == f32   ? AFHIP_PRECISION_F32
                                   : x.type == f16 ? AFHIP_PRECISION_F16
                                                   : AFHIP_PRECISION_BF16);
    const int cus = device_cus();
    const long long need = gather || !own || (wg && wg[0] == '0')
                               ? 0
                               : nn_wgemm_workspace(x.type, g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, cus);
    const bool rows = need <= 0 || (!(wg && wg[0] == '1') && rows_by_rule(x, g) &&
                                    afhip_k_conv2_nn_wgrad_rows_workspace(x.type, precision, g.x.d, g.w.d, g.y.d, g.st,
                                                                          g.pd, g.dl) > 0);
    const auto others = [&] { wgrad_rows_or_gather(dy, x, g, precision, out_type, o, gather); };
    if (rows) {
        others();
        return;
    }
    or_with_less_memory(
        [&] {
            auto ws = scratch((size_t)need);
            check_k(nn_wgemm(x.type, out_type, o, x.data(), dy.data(), g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl, cus,
                             ws->ptr, need, stream()),
                    "convolve2_gradient_nn");
        },
        others);
}

// cpu::conv2FilterGradient<T>, src/backend/cpu/convolve.cpp:213-243
static af_array conv2_filter_grad(const ArrayImpl &dy, const ArrayImpl &x, const ArrayImpl &w,
                                  const NNGeom &g, int precision, af_dtype out_type) {
    NewHandle out(make_handle(out_type, g.w));
    if (g.w.elements() == 0) return out.release();
    void *o = out.data();
    if (dy.elements() == 0 || g.x.elements() == 0) {
        check_k(afhip_k_fill(out_type, o, 0.0, g.w.elements(), stream()), "fill");
        return out.release();
    }
    if (x.type == f64) {
        check_k(afhip_k_conv2_nn_f64(2, o, x.data(), dy.data(), g.x.d, g.w.d, g.y.d, g.st, g.pd, g.dl,
                                     stream()),
                "convolve2_gradient_nn");
        return out.release();
    }
    run_wgrad(dy, x, g, precision, out_type, o);
    return out.release();
}

// Frequency-domain convolution (src/backend/cpu/fftconvolve.cpp:42-203 and
// the fallback of src/api/c/fftconvolve.cpp:52-121). The batched path takes
// the filter converted to the signal's type (castArray<T>: fractional taps on
// an integer signal truncate); the fallback (DIFF batches, complex signals)
// converts it straight to the complex compute type.
static af_array fft_convolve(const ArrayImpl &sig, const ArrayImpl &filt, BatchKind kind, int rank,
                             bool expand) {
    const bool fallback = kind == BATCH_DIFF || sig.type == c32 || sig.type == c64;
    std::shared_ptr<Buffer> fb;
    af_dtype ft;
    if (fallback) {
        ft = (filt.type == f16 || filt.type == afhip_bf16) ? f32 : filt.type;
        fb = cast_buffer(filt, ft);
    } else {
        ft = sig.type;
        fb = cast_buffer(filt, ft);
    }
    dim4 od;
    if (kind == BATCH_DIFF) {
        // base dims as the batched kinds; dims past the rank: max(s, f)
        // (odims of src/api/c/fftconvolve.cpp:72-97)
        for (int d = 0; d < AF_MAX_DIMS; ++d)
            od[d] = d < rank ? (expand ? sig.dims[d] + filt.dims[d] - 1 : sig.dims[d])
                             : std::max(sig.dims[d], filt.dims[d]);
    } else {
        od = conv_out_dims(sig.dims, filt.dims, kind, rank, expand);
    }
    NewHandle out(make_handle(sig.type, od));
    if (od.elements() == 0) return out.release();
    const long long need =
        afhip_k_fft_convolve_workspace(sig.type, sig.dims.d, filt.dims.d, od.d, (int)kind, rank);
    if (need < 0) AFHIP_THROW(AF_ERR_SIZE, "fft_convolve: a padded axis exceeds 2^24 elements");
    auto ws = scratch((size_t)need);
    check_k(afhip_k_fft_convolve(sig.type, out.data(), od.d, sig.data(), sig.dims.d, ft, fb->ptr,
                                 filt.dims.d, (int)kind, rank, expand ? 1 : 0, ws->ptr, need, stream()),
            "fft_convolve");
    return out.release();
}

// Scalar/scalar separable filters on a complex signal (src/api/c/convolve.cpp:57-68
// with accT = cfloat / cdouble): y = x * (c * r), the filter product formed in
// accT with each real product rounded before the sum, as std::complex does.
template <typename R>
static void cmul(const R *a, const R *b, R *o) {
#pragma clang fp contract(off)
    o[0] = a[0] * b[0] - a[1] * b[1];
    o[1] = a[0] * b[1] + a[1] * b[0];
}

static af_array scale_complex(const ArrayImpl &sig, const std::shared_ptr<Buffer> &cb,
                              const std::shared_ptr<Buffer> &rb, af_dtype at) {
    double re, im;
    if (at == c32) {
        float c[2], r[2], p[2];
        check_hip(hipMemcpyAsync(c, cb->ptr, 8, hipMemcpyDeviceToHost, stream()), "copy");
        check_hip(hipMemcpyAsync(r, rb->ptr, 8, hipMemcpyDeviceToHost, stream()), "copy");
        sync_stream();
        cmul(c, r, p);
        re = p[0];
        im = p[1];
    } else {
        double c[2], r[2], p[2];
        check_hip(hipMemcpyAsync(c, cb->ptr, 16, hipMemcpyDeviceToHost, stream()), "copy");
        check_hip(hipMemcpyAsync(r, rb->ptr, 16, hipMemcpyDeviceToHost, stream()), "copy");
        sync_stream();
        cmul(c, r, p);
        re = p[0];
        im = p[1];
    }
    NewHandle o(make_handle(sig.type, sig.dims));
    check_k(afhip_k_scale_complex(sig.type, o.data(), sig.data(), re, im, sig.elements(), stream()),
            "convolve2_sep");
    return o.release();
}

}  // namespace detail

// ---------------------------------------------------------------- C API
// src/api/c/convolve.cpp:132-215
static af_err convolve_common(af_array *out, const af_array signal, const af_array filter,
                              const af_conv_mode mode, const int rank) {
    try {
        const ArrayImpl &s = get(signal);
        const ArrayImpl &f = get(filter);
        ARG_ASSERT(0, out != nullptr);
        if (f.dims.ndims() == 0 || s.dims.ndims() == 0) return af_retain_array(out, signal);
        const BatchKind kind = identify_batch_kind(rank, s.dims, f.dims);
        ARG_ASSERT(1, kind != BATCH_UNSUPPORTED && kind != BATCH_DIFF);
        const bool expand = mode == AF_CONV_EXPAND;
        (void)acc_type(s.type);  // TYPE_ERROR(1, stype) for f16 / bf16
        af_array o = detail::convolve(s, f, kind, rank, expand);
        *out = o;
    }
    CATCHALL;
    return AF_SUCCESS;
}

// src/api/c/fftconvolve.cpp:162-219: batch kind, dtype dispatch (every
// dtype but f16), then the batched path or, for DIFF batches and complex
// signals, the fallback (:52-121).
static af_err fft_convolve_common(af_array *out, const af_array signal, const af_array filter,
                                  const bool expand, const int rank) {
    try {
        const ArrayImpl &s = get(signal);
        const ArrayImpl &f = get(filter);
        ARG_ASSERT(0, out != nullptr);
        const BatchKind kind = identify_batch_kind(rank, s.dims, f.dims);
        ARG_ASSERT(1, kind != BATCH_UNSUPPORTED);
        (void)acc_type(s.type);  // TYPE_ERROR(1, stype) for f16 / bf16
        *out = detail::fft_convolve(s, f, kind, rank, expand);
    }
    CATCHALL;
    return AF_SUCCESS;
}

}  // namespace afhip

using namespace afhip;

extern "C" {

// src/api/c/fftconvolve.cpp:247-264
AFAPI af_err af_fft_convolve1(af_array *out, const af_array signal, const af_array filter,
                              const af_conv_mode mode) {
    return fft_convolve_common(out, signal, filter, mode == AF_CONV_EXPAND, 1);
}
AFAPI af_err af_fft_convolve2(af_array *out, const af_array signal, const af_array filter,
                              const af_conv_mode mode) {
    try {
        if (get(signal).dims.ndims() < 2 && get(filter).dims.ndims() < 2)
            return fft_convolve_common(out, signal, filter, mode == AF_CONV_EXPAND, 1);
        return fft_convolve_common(out, signal, filter, mode == AF_CONV_EXPAND, 2);
    }
    CATCHALL;
}
AFAPI af_err af_fft_convolve3(af_array *out, const af_array signal, const af_array filter,
                              const af_conv_mode mode) {
    try {
        if (get(signal).dims.ndims() < 3 && get(filter).dims.ndims() < 3)
            return fft_convolve_common(out, signal, filter, mode == AF_CONV_EXPAND, 2);
        return fft_convolve_common(out, signal, filter, mode == AF_CONV_EXPAND, 3);
    }
    CATCHALL;
}

// src/api/c/convolve.cpp:217-226
AFAPI af_err af_convolve1(af_array *out, const af_array signal, const af_array filter,
                          const af_conv_mode mode, af_conv_domain domain) {
    try {
        if (is_freq_domain(1, get(signal).dims, get(filter).dims, domain))
            return af_fft_convolve1(out, signal, filter, mode);
        return convolve_common(out, signal, filter, mode, 1);
    }
    CATCHALL;
}

// src/api/c/convolve.cpp:228-241
AFAPI af_err af_convolve2(af_array *out, const af_array signal, const af_array filter,
                          const af_conv_mode mode, af_conv_domain domain) {
    try {
        if (get(signal).dims.ndims() < 2 || get(filter).dims.ndims() < 2)
            return af_convolve1(out, signal, filter, mode, domain);
        if (is_freq_domain(2, get(signal).dims, get(filter).dims, domain))
            return af_fft_convolve2(out, signal, filter, mode);
        return convolve_common(out, signal, filter, mode, 2);
    }
    CATCHALL;
}

// src/api/c/convolve.cpp:243-256
AFAPI af_err af_convolve3(af_array *out, const af_array signal, const af_array filter,
                          const af_conv_mode mode, af_conv_domain domain) {
    try {
        if (get(signal).dims.ndims() < 3 || get(filter).dims.ndims() < 3)
            return af_convolve2(out, signal, filter, mode, domain);
        if (is_freq_domain(3, get(signal).dims, get(filter).dims, domain))
            return af_fft_convolve3(out, signal, filter, mode);
        return convolve_common(out, signal, filter, mode, 3);
    }
    CATCHALL;
}

// isVector, src/backend/common/ArrayInfo.cpp:122-130
static bool is_vector(const dim4 &d) {
    int singular = 0, nonsingular = 0;
    for (int i = 0; i < AF_MAX_DIMS; ++i) {
        nonsingular += (d[i] != 0 && d[i] != 1);
        singular += (d[i] == 1);
    }
    return singular == AF_MAX_DIMS - 1 && nonsingular == 1;
}

// src/api/c/convolve.cpp:258-334 and :50-75
AFAPI af_err af_convolve2_sep(af_array *out, const af_array col_filter, const af_array row_filter,
                              const af_array signal, const af_conv_mode mode) {
    try {
        const ArrayImpl &s = get(signal);
        ARG_ASSERT(1, s.dims.ndims() >= 2);
        ARG_ASSERT(0, out != nullptr);
        const af_dtype at = acc_type(s.type);
        const bool expand = mode == AF_CONV_EXPAND;
        const ArrayImpl &cf = get(col_filter);
        const ArrayImpl &rf = get(row_filter);
        auto cb = cast_buffer(cf, at);
        auto rb = cast_buffer(rf, at);
        if (cf.elements() == 1 && rf.elements() == 1) {
            // scalar/scalar: y = T(accT(x) * (c * r))
            if (at == c32 || at == c64) {
                *out = detail::scale_complex(s, cb, rb, at);
                return AF_SUCCESS;
            }
            if (at != f32 && at != f64) TYPE_ERROR(1, s.type);
            double scale;
            if (at == f32) {
                float c = 0, r = 0;
                check_hip(hipMemcpyAsync(&c, cb->ptr, 4, hipMemcpyDeviceToHost, stream()), "copy");
                check_hip(hipMemcpyAsync(&r, rb->ptr, 4, hipMemcpyDeviceToHost, stream()), "copy");
                sync_stream();
                scale = (double)(c * r);
            } else {
                double c = 0, r = 0;
                check_hip(hipMemcpyAsync(&c, cb->ptr, 8, hipMemcpyDeviceToHost, stream()), "copy");
                check_hip(hipMemcpyAsync(&r, rb->ptr, 8, hipMemcpyDeviceToHost, stream()), "copy");
                sync_stream();
                scale = c * r;
            }
            NewHandle o(make_handle(s.type, s.dims));
            check_k(afhip_k_scale(s.type, o.data(), s.data(), scale, s.elements(), stream()),
                    "convolve2_sep");
            *out = o.release();
            return AF_SUCCESS;
        }
        ARG_ASSERT(2, is_vector(cf.dims));
        ARG_ASSERT(3, is_vector(rf.dims));
        *out = detail::convolve2_sep(s, cb, cf.elements(), rb, rf.elements(), expand);
    }
    CATCHALL;
    return AF_SUCCESS;
}

static af_err nn_forward(af_array *out, const af_array signal, const af_array filter,
                         const unsigned stride_dims, const dim_t *strides,
                         const unsigned padding_dims, const dim_t *paddings,
                         const unsigned dilation_dims, const dim_t *dilations, int precision,
                         af_dtype out_type) {
    try {
        const ArrayImpl &s = get(signal);
        const ArrayImpl &f = get(filter);
        ARG_ASSERT(0, out != nullptr);
        dim4 stride(stride_dims, strides), padding(padding_dims, paddings),
            dilation(dilation_dims, dilations);
        const dim_t sn = stride.ndims(), pn = padding.ndims(), dn = dilation.ndims();
        ARG_ASSERT(3, sn > 0 && sn <= 2);
        ARG_ASSERT(5, pn >= 0 && pn <= 2);
        ARG_ASSERT(7, dn > 0 && dn <= 2);
        DIM_ASSERT(1, s.dims[2] == f.dims[2]);
        const af_dtype t = s.type;
        if (t != f32 && t != f64 && t != f16 && t != afhip_bf16) TYPE_ERROR(1, t);
        if (f.type != t) AFHIP_THROW(AF_ERR_INTERNAL, "Invalid type for input array.");
        const af_dtype ot = detail::nn_out_type(t, out_type);
        if (t == f64) {
            ARG_ASSERT(9, precision == AFHIP_PRECISION_DEFAULT);
            if (ot != f64) TYPE_ERROR(10, ot);
        }
        auto g = detail::nn_geom(s.dims, f.dims, stride, padding, dilation);
        detail::check_nn_geom(g);
        *out = detail::conv2_nn(s, f, g, precision, ot);
    }
    CATCHALL;
    return AF_SUCCESS;
}

// src/api/c/convolve.cpp:344-392
AFAPI af_err af_convolve2_nn(af_array *out, const af_array signal, const af_array filter,
                             const unsigned stride_dims, const dim_t *strides,
                             const unsigned padding_dims, const dim_t *paddings,
                             const unsigned dilation_dims, const dim_t *dilations) {
    return nn_forward(out, signal, filter, stride_dims, strides, padding_dims, paddings, dilation_dims,
                      dilations, AFHIP_PRECISION_DEFAULT, (af_dtype)-1);
}

AFAPI af_err afhip_convolve2_nn_ex(af_array *out, const af_array signal, const af_array filter,
                                   const unsigned stride_dims, const dim_t *strides,
                                   const unsigned padding_dims, const dim_t *paddings,
                                   const unsigned dilation_dims, const dim_t *dilations,
                                   afhip_precision precision, af_dtype out_type) {
    return nn_forward(out, signal, filter, stride_dims, strides, padding_dims, paddings, dilation_dims,
                      dilations, (int)precision, out_type);
}

static af_err nn_gradient(af_array *out, const af_array incoming_gradient,
                          const af_array original_signal, const af_array original_filter,
                          const af_array convolved_output, const unsigned stride_dims,
                          const dim_t *strides, const unsigned padding_dims, const dim_t *paddings,
                          const unsigned dilation_dims, const dim_t *dilations,
                          af_conv_gradient_type grad_type, int precision, af_dtype out_type,
                          bool strict_types) {
    try {
        const ArrayImpl &g = get(incoming_gradient);
        const ArrayImpl &s = get(original_signal);
        const ArrayImpl &f = get(original_filter);
        const ArrayImpl &o = get(convolved_output);
        ARG_ASSERT(0, out != nullptr);
        // src/api/c/convolve.cpp:434-437
        DIM_ASSERT(1, g.dims == o.dims);
        DIM_ASSERT(3, o.dims[2] == f.dims[3]);
        DIM_ASSERT(3, o.dims[3] == s.dims[3]);
        DIM_ASSERT(2, s.dims[2] == f.dims[2]);
        dim4 stride(stride_dims, strides), padding(padding_dims, paddings),
            dilation(dilation_dims, dilations);
        const dim_t sn = stride.ndims(), pn = padding.ndims(), dn = dilation.ndims();
        ARG_ASSERT(3, sn > 0 && sn <= 2);
        ARG_ASSERT(5, pn >= 0 && pn <= 2);
        ARG_ASSERT(7, dn > 0 && dn <= 2);
        // The reference takes T from convolved_output and requires all four
        // arrays to be T (src/api/c/convolve.cpp:452, handle.hpp:53-54). The
        // extension entry point reads only the dims of convolved_output (it
        // may hold the FP32 output of a BF16 forward), so T comes from the
        // incoming gradient there.
        const af_dtype t = strict_types ? o.type : g.type;
        if (t != f32 && t != f64 && t != f16 && t != afhip_bf16) TYPE_ERROR(1, t);
        if (g.type != t || s.type != t || f.type != t || (strict_types && o.type != t))
            AFHIP_THROW(AF_ERR_INTERNAL, "Invalid type for input array.");
        const af_dtype ot = detail::nn_out_type(t, out_type);
        if (t == f64) {
            ARG_ASSERT(12, precision == AFHIP_PRECISION_DEFAULT);
            if (ot != f64) TYPE_ERROR(13, ot);
        }
        auto geo = detail::nn_geom(s.dims, f.dims, stride, padding, dilation);
        detail::check_nn_geom(geo);
        // The incoming gradient must have the forward output's shape for the
        // kernels' indexing (the reference reads it through the same dims).
        DIM_ASSERT(1, g.dims == geo.y);
        if (grad_type == AF_CONV_GRADIENT_FILTER)
            *out = detail::conv2_filter_grad(g, s, f, geo, precision, ot);
        else
            *out = detail::conv2_data_grad(g, s, f, geo, precision, ot);
    }
    CATCHALL;
    return AF_SUCCESS;
}

// src/api/c/convolve.cpp:394-477
AFAPI af_err af_convolve2_gradient_nn(af_array *out, const af_array incoming_gradient,
                                      const af_array original_signal, const af_array original_filter,
                                      const af_array convolved_output, const unsigned stride_dims,
                                      const dim_t *strides, const unsigned padding_dims,
                                      const dim_t *paddings, const unsigned dilation_dims,
                                      const dim_t *dilations, af_conv_gradient_type grad_type) {
    return nn_gradient(out, incoming_gradient, original_signal, original_filter, convolved_output,
                       stride_dims, strides, padding_dims, paddings, dilation_dims, dilations,
                       grad_type, AFHIP_PRECISION_DEFAULT, (af_dtype)-1, true);
}

AFAPI af_err afhip_convolve2_gradient_nn_ex(
    af_array *out, const af_array incoming_gradient, const af_array original_signal,
    const af_array original_filter, const af_array convolved_output, const unsigned stride_dims,
    const dim_t *strides, const unsigned padding_dims, const dim_t *paddings,
    const unsigned dilation_dims, const dim_t *dilations, af_conv_gradient_type grad_type,
    afhip_precision precision, af_dtype out_type) {
    return nn_gradient(out, incoming_gradient, original_signal, original_filter, convolved_output,
                       stride_dims, strides, padding_dims, paddings, dilation_dims, dilations,
                       grad_type, (int)precision, out_type, false);
}

}  // extern "C"

struct afhip_nn_step_plan_t {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<void *> kept;                            // workspaces the graph uses
    std::vector<std::shared_ptr<afhip::Buffer>> arrays;  // x, w, dy, y, dx, dw
    ~afhip_nn_step_plan_t() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (void *p : kept) afhip::pool_free(p);
    }
};

extern "C" {

// The three passes of one step through the public entry points (checks,
// dispatch, allocation); the handles are released on failure.
static af_err nn_step_passes(af_array *y, af_array *dx, af_array *dw, const af_array x, const af_array w,
                             const af_array dy, const unsigned sdims, const dim_t *strides, const unsigned pdims,
                             const dim_t *paddings, const unsigned ddims, const dim_t *dilations, int precision,
                             af_dtype out_type) {
    *y = *dx = *dw = nullptr;
    af_err e = nn_forward(y, x, w, sdims, strides, pdims, paddings, ddims, dilations, precision, out_type);
    if (e == AF_SUCCESS)
        e = nn_gradient(dx, dy, x, w, *y, sdims, strides, pdims, paddings, ddims, dilations,
                        AF_CONV_GRADIENT_DATA, precision, out_type, false);
    if (e == AF_SUCCESS)
        e = nn_gradient(dw, dy, x, w, *y, sdims, strides, pdims, paddings, ddims, dilations,
                        AF_CONV_GRADIENT_FILTER, precision, out_type, false);
    if (e != AF_SUCCESS) {
        for (af_array *h : {y, dx, dw})
            if (*h) {
                destroy_handle(*h);
                *h = nullptr;
            }
    }
    return e;
}

AFAPI af_err afhip_nn_step_plan_create(afhip_nn_step_plan *plan, af_array *y, af_array *dx, af_array *dw,
                                       const af_array x, const af_array w, const af_array dy,
                                       const unsigned stride_dims, const dim_t *strides,
                                       const unsigned padding_dims, const dim_t *paddings,
                                       const unsigned dilation_dims, const dim_t *dilations,
                                       afhip_precision precision, af_dtype out_type) {
    try {
        ARG_ASSERT(0, plan != nullptr && y != nullptr && dx != nullptr && dw != nullptr);
        // eager run: argument checks, first-use kernel setup, pool warm-up
        af_array e[3];
        af_err rc = nn_step_passes(&e[0], &e[1], &e[2], x, w, dy, stride_dims, strides, padding_dims, paddings,
                                   dilation_dims, dilations, (int)precision, out_type);
        if (rc != AF_SUCCESS) return rc;
        for (af_array h : e) destroy_handle(h);
        sync_stream();

        auto p = std::make_unique<afhip_nn_step_plan_t>();
        af_array h[3] = {nullptr, nullptr, nullptr};
        hipStream_t s = stream();
        check_hip(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed), "hipStreamBeginCapture");
        pool_keep(&p->kept);
        rc = nn_step_passes(&h[0], &h[1], &h[2], x, w, dy, stride_dims, strides, padding_dims, paddings,
                            dilation_dims, dilations, (int)precision, out_type);
        pool_keep(nullptr);
        const hipError_t ce = hipStreamEndCapture(s, &p->graph);
        if (rc != AF_SUCCESS || ce != hipSuccess) {
            for (af_array a : h)
                if (a) destroy_handle(a);
            if (rc != AF_SUCCESS) return rc;
            check_hip(ce, "hipStreamEndCapture");
        }
        const hipError_t ie = hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0);
        if (ie != hipSuccess) {
            for (af_array a : h) destroy_handle(a);
            check_hip(ie, "hipGraphInstantiate");
        }
        for (af_array a : {x, w, dy}) p->arrays.push_back(get(a).buf);
        for (af_array a : h) p->arrays.push_back(get(a).buf);
        *y = h[0];
        *dx = h[1];
        *dw = h[2];
        *plan = p.release();
    }
    CATCHALL;
    return AF_SUCCESS;
}

AFAPI af_err afhip_nn_step_plan_run(afhip_nn_step_plan plan) {
    try {
        ARG_ASSERT(0, plan != nullptr);
        check_hip(hipGraphLaunch(plan->exec, stream()), "hipGraphLaunch");
    }
    CATCHALL;
    return AF_SUCCESS;
}

AFAPI af_err afhip_nn_step_plan_release(afhip_nn_step_plan plan) {
    try {
        if (plan) {
            sync_stream();  // a replay in flight still uses the workspaces
            delete plan;
        }
    }
    CATCHALL;
    return AF_SUCCESS;
}

// include/af/data.h:515
AFAPI af_err af_constant(af_array *arr, const double val, const unsigned ndims,
                         const dim_t *const dims, const af_dtype type) {
    try {
        ARG_ASSERT(0, arr != nullptr);
        ARG_ASSERT(2, ndims >= 1 && ndims <= 4);
        if (!dtype_known(type)) TYPE_ERROR(4, type);
        dim4 d(ndims, dims);
        NewHandle o(make_handle(type, d));
        if (d.elements() > 0)
            check_k(afhip_k_fill(type, o.data(), val, d.elements(), stream()), "af_constant");
        *arr = o.release();
    }
    CATCHALL;
    return AF_SUCCESS;
}

// include/af/arith.h (af_cast)
AFAPI af_err af_cast(af_array *out, const af_array in, const af_dtype type) {
    try {
        ARG_ASSERT(0, out != nullptr);
        const ArrayImpl &a = get(in);
        if (!dtype_known(type)) TYPE_ERROR(2, type);
        if (a.type == type) return af_retain_array(out, in);
        NewHandle o(make_handle(type, a.dims));
        if (a.elements() > 0)
            check_k(afhip_k_cast(type, o.data(), a.type, a.data(), a.elements(), stream()),
                    "af_cast");
        *out = o.release();
    }
    CATCHALL;
    return AF_SUCCESS;
}

}  // extern "C"
