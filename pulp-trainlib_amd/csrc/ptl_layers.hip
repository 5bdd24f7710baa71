// Conv2D, pointwise convolution and Linear: forward, weight-gradient and
// input-gradient steps expressed as index maps over the MFMA GEMM
// (ptl_gemm.hip).  Nothing here moves data: each step is one GEMM launch
// (plus a split-K reduction where the output is too small to fill the chip)
// reading the caller's tensors in place.
//
// Batched mode stores `ns` samples back to back (sample stride = blob->dim);
// the sample index is folded into the pixel axis of the GEMM for forward and
// input gradient, and into the contraction axis for the weight gradient, so
// the sum over samples happens in the fp32 accumulator.
#include "ptl_common.hpp"
#include "ptl_host.hpp"
#include "ptl_conv_tile.hpp"
#include "ptl_sum.hpp"

#define STEP_BW_BOTH 3  // weight and input gradient together (library-internal step code)
#include "ptl_api.h"
#include "ptl_internal.h"

#include <stdio.h>
#include <algorithm>

namespace ptl {

// ---- small kernels -----------------------------------------------------------

// Zero-stuffed copy of an output gradient for strided convolutions:
// dst[b][c][ho*sh][wo*sw] = src[b][c][ho][wo] (CHW) or the HWC equivalent.
// One workgroup per plane (CHW: a channel of a sample, HWC: a sample): it clears the plane, then scatters the
// source elements into it (one division per source element instead of five per destination element).
template <typename T>
__global__ __launch_bounds__(256) void dilate_kernel(const T *__restrict__ src, T *__restrict__ dst, int Ho, int Wo,
                                                     int Hd, int Wd, int sh, int sw, int cin) {
    // cin = innermost channel count (1 for CHW planes, C for HWC)
    const unsigned n = (unsigned)Hd * Wd * cin, m = (unsigned)Ho * Wo * cin, rowlen = (unsigned)Wo * cin;
    const T *sp = src + (size_t)blockIdx.x * m;
    T *dp = dst + (size_t)blockIdx.x * n;
    for (unsigned i = threadIdx.x; i < n; i += 256) dp[i] = (T)0;
    __syncthreads();  // orders the two writes of a position within the workgroup
    for (unsigned i = threadIdx.x; i < m; i += 256) {
        const unsigned ho = i / rowlen, r = i - ho * rowlen;
        const unsigned wo = cin == 1 ? r : r / cin, c = cin == 1 ? 0 : r - wo * cin;
        dp[((ho * sh) * Wd + wo * sw) * cin + c] = sp[i];
    }
}

// dst[0 .. n) = 0, 16 bytes per thread where the alignment allows.
template <typename T>
__global__ __launch_bounds__(256) void zero_kernel(T *__restrict__ dst, size_t n, int vec) {
    constexpr int VEC = 16 / (int)sizeof(T);
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (vec) {
        if (i * VEC + VEC <= n) reinterpret_cast<uint4 *>(dst)[i] = make_uint4(0, 0, 0, 0);
        else
            for (size_t e = i * VEC; e < n; ++e) dst[e] = (T)0;
    } else if (i < n) {
        dst[i] = (T)0;
    }
}

// out[b][c][pix] += bias[c] (CHW) or out[b][pix][c] += bias[c] (HWC: inner = 1): a thread adds to one 16-byte piece, the
// elements of which start at channel and position of the first and walk on (element by element and with a 64-bit
// division each it took 16 us for 7.6 M elements in fp16, 4.9 this way).  `total` <= 2^30 elements, the first of which has
// channel c0 and position p0 < 2^31: every index fits 32 bits.
constexpr size_t BIAS_ADD_MOST = (size_t)1 << 30;
template <typename T>
__global__ __launch_bounds__(256) void bias_add_kernel(T *__restrict__ out, const T *__restrict__ bias, unsigned total,
                                                       unsigned C, unsigned inner, unsigned c0, unsigned p0) {
    constexpr unsigned V = 16 / sizeof(T);
    const unsigned i0 = (blockIdx.x * 256 + threadIdx.x) * V;
    if (i0 >= total) return;
    unsigned q = (p0 + i0) / inner, p = p0 + i0 - q * inner, c = (c0 + q) % C;
    T v[V];
    const bool whole = i0 + V <= total;
    if (whole) __builtin_memcpy(v, out + i0, 16);
#pragma unroll
    for (unsigned e = 0; e < V; ++e) {
        if (whole) v[e] = (T)((float)v[e] + (float)bias[c]);
        else if (i0 + e < total) out[i0 + e] = (T)((float)out[i0 + e] + (float)bias[c]);
        if (++p == inner) {
            p = 0;
            c = c + 1 == C ? 0 : c + 1;
        }
    }
    if (whole) __builtin_memcpy(out + i0, v, 16);
}

// part[s][c] = sum of dY over the positions of share s: channel-major tensors give a workgroup a channel and a share of
// its (sample, position) axis, read in 16-byte pieces inside each sample.
template <typename T>
__global__ __launch_bounds__(256) void bias_grad_kernel(const T *__restrict__ dy, float *__restrict__ part, T *__restrict__ db,
                                                        int ns, int C, int pix, int per_share) {
    constexpr int V = 16 / (int)sizeof(T);
    const int c = blockIdx.x, b0 = blockIdx.y * per_share, b1 = min(ns, b0 + per_share);
    const int pieces = (pix + V - 1) / V;  // per sample
    LongSum<T> s;
    s.clear();
    for (int i = threadIdx.x; i < (b1 - b0) * pieces; i += 256) {
        const int b = i / pieces, p = (i - b * pieces) * V;
        const T *src = dy + ((size_t)(b0 + b) * C + c) * pix + p;
        if (p + V <= pix) {
            T v[V];
            __builtin_memcpy(v, src, 16);
#pragma unroll
            for (int e = 0; e < V; ++e) s.add((float)v[e]);
        } else {
            for (int e = 0; p + e < pix; ++e) s.add((float)src[e]);
        }
    }
    __shared__ LongSum<T> red[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s.fold(o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < 4; ++w) s.add(red[w]);
        if (gridDim.y == 1) db[c] = (T)s.value();
        else part[(size_t)blockIdx.y * C + c] = s.value();
    }
}

// The same for tensors with the channels innermost (and for batches of vectors): a workgroup owns 64 channels and a share
// of the rows, four rows at a time with four loads in flight.
template <typename T>
__global__ __launch_bounds__(256) void bias_grad_rows_kernel(const T *__restrict__ dy, float *__restrict__ part, T *__restrict__ db,
                                                             int rows, int C, int per_share) {
    const int o = threadIdx.x & 63, w = threadIdx.x >> 6, c = blockIdx.x * 64 + o;
    const int r0 = blockIdx.y * per_share, r1 = min(rows, r0 + per_share);
    LongSum<T> s;
    s.clear();
    if (c < C) {
        int r = r0 + w;
        for (; r + 12 < r1; r += 16) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = (float)dy[(size_t)(r + 4 * u) * C + c];
#pragma unroll
            for (int u = 0; u < 4; ++u) s.add(v[u]);
        }
        for (; r < r1; r += 4) s.add((float)dy[(size_t)r * C + c]);
    }
    __shared__ LongSum<T> red[4][64];
    red[w][o] = s;
    __syncthreads();
    if (w == 0 && c < C) {
#pragma unroll
        for (int q = 1; q < 4; ++q) s.add(red[q][o]);
        if (gridDim.y == 1) db[c] = (T)s.value();
        else part[(size_t)blockIdx.y * C + c] = s.value();
    }
}

// db[c] = sum of dY over samples and positions: one launch where the channels alone fill the chip or little is to be read,
// else shares of it and their sum (45 channels of 27 753 positions in fp32: 37.6 us with one workgroup per channel and a
// 64-bit division per element, 8.5 this way).
template <typename T>
static int bias_grad(const T *dy, T *db, int ns, int C, int pix, int hwc) {
    State &st = state();
    const bool by_rows = hwc || pix == 1;
    const long long rows = (long long)ns * pix, units = by_rows ? rows : ns, wide = by_rows ? (C + 63) / 64 : C;
    // a share is worth a launch only if it shortens the walk of a workgroup by a good deal
    const long long walk = by_rows ? rows / 16 : rows / (256 * (16 / (long long)sizeof(T)));
    long long shares = 1;
    if (walk > 32) shares = (2ll * st.num_cu + wide - 1) / wide;
    if (shares > units) shares = units;
    if (shares > (walk + 7) / 8) shares = (walk + 7) / 8;
    if (shares < 1) shares = 1;
    const long long per = (units + shares - 1) / shares;
    shares = (units + per - 1) / per;
    float *part = nullptr;
    if (shares > 1 && !(part = workspace((size_t)shares * C * sizeof(float)))) return 2;
    if (by_rows)
        hipLaunchKernelGGL((bias_grad_rows_kernel<T>), dim3((unsigned)wide, (unsigned)shares), dim3(256), 0, st.stream, dy, part, db,
                           (int)rows, C, (int)per);
    else
        hipLaunchKernelGGL((bias_grad_kernel<T>), dim3(C, (unsigned)shares), dim3(256), 0, st.stream, dy, part, db, ns, C, pix, (int)per);
    if (shares > 1) launch_share_sum<T>(part, db, C, (int)shares, st.stream);
    return hip_ok(hipGetLastError(), "bias grad launch") ? 0 : 2;
}

// (a matrix may have up to 2^62 elements: one launch for each 2^30 of them)
template <typename T>
static void launch_bias_add(T *out, const T *bias, size_t total, int C, int inner) {
    constexpr size_t V = 16 / sizeof(T);
    for (size_t at = 0; at < total; at += BIAS_ADD_MOST) {
        const size_t n = total - at < BIAS_ADD_MOST ? total - at : BIAS_ADD_MOST, q = at / inner;
        hipLaunchKernelGGL((bias_add_kernel<T>), dim3((unsigned)((n + 256 * V - 1) / (256 * V))), dim3(256), 0, state().stream,
                           out + at, bias, (unsigned)n, (unsigned)C, (unsigned)inner, (unsigned)(q % C), (unsigned)(at - q * inner));
    }
}

static inline unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

static bool fits_int(size_t v) { return v < ((size_t)1 << 31); }

// ---- Conv2D ----------------------------------------------------------------------

struct ConvGeom {
    int Ci, H, W, Co, Ho, Wo, Hk, Wk;
    int Up, Dp, Lp, Rp, sh, sw;
    int hwc;
};

template <typename Args>
static int conv_geom(const Args *a, ConvGeom &g, const char *fn, bool need_divisible) {
    if (!a || !a->input || !a->coeff || !a->output) {
        printf("[%s:] null argument structure\n", fn);
        set_error("%s: null argument structure", fn);
        return 1;
    }
    g.Ci = a->input->C;
    g.H = a->input->H;
    g.W = a->input->W;
    g.Co = a->output->C;
    g.Ho = a->output->H;
    g.Wo = a->output->W;
    g.Hk = a->coeff->H;
    g.Wk = a->coeff->W;
    g.Up = a->Upad;
    g.Dp = a->Dpad;
    g.Lp = a->Lpad;
    g.Rp = a->Rpad;
    g.sh = a->stride_h;
    g.sw = a->stride_w;
    g.hwc = a->HWC;
    if (a->USE_IM2COL != 0 && a->USE_IM2COL != 1) {
        printf("[%s:] Invalid selection of the conv2d algorithm (im2col or not)\n", fn);
        set_error("%s: USE_IM2COL must be 0 or 1", fn);
        return 1;
    }
    if (g.hwc != 0 && g.hwc != 1) {
        printf("[%s:] Invalid data layout format (HWC or CHW)!\n", fn);
        set_error("%s: HWC must be 0 or 1", fn);
        return 1;
    }
    if (a->USE_IM2COL == 0 && g.hwc == 1) {
        printf("[%s:] Naive kernel for HWC Conv2D not implemented!\n", fn);
        set_error("%s: naive HWC Conv2D does not exist in the reference", fn);
        return 1;
    }
    if (g.Ci <= 0 || g.H <= 0 || g.W <= 0 || g.Co <= 0 || g.Hk <= 0 || g.Wk <= 0 || g.sh <= 0 || g.sw <= 0 ||
        g.Up < 0 || g.Dp < 0 || g.Lp < 0 || g.Rp < 0) {
        printf("[%s:] invalid tensor geometry\n", fn);
        set_error("%s: invalid tensor geometry", fn);
        return 1;
    }
    int nh = g.H - g.Hk + g.Up + g.Dp, nw = g.W - g.Wk + g.Lp + g.Rp;
    if (nh < 0 || nw < 0) {
        printf("[%s:] kernel larger than padded input\n", fn);
        set_error("%s: kernel larger than padded input", fn);
        return 1;
    }
    if (need_divisible && a->USE_IM2COL == 1) {
        if ((nh + g.sh) % g.sh > 0) {
            printf("\n[pulp_im2col] Invalid H stride (non multiple H sizes): have H_in=%d, H_ker=%d, U_pad=%d, "
                   "D_pad=%d, H_stride=%d, remainder=%d",
                   g.H, g.Hk, g.Up, g.Dp, g.sh, (nh + g.sh) % g.sh);
            set_error("%s: H stride does not divide the padded extent", fn);
            return 1;
        }
        if ((nw + g.sw) % g.sw > 0) {
            printf("\n[pulp_im2col] Invalid W stride (non multiple W sizes): have W_in=%d, W_ker=%d, L_pad=%d, "
                   "R_pad=%d, W_stride=%d, remainder=%d",
                   g.W, g.Wk, g.Lp, g.Rp, g.sw, (nw + g.sw) % g.sw);
            set_error("%s: W stride does not divide the padded extent", fn);
            return 1;
        }
    }
    if (g.Ho != nh / g.sh + 1 || g.Wo != nw / g.sw + 1) {
        printf("[%s:] output blob is %dx%d but the geometry gives %dx%d\n", fn, g.Ho, g.Wo, nh / g.sh + 1,
               nw / g.sw + 1);
        set_error("%s: output blob size does not match the convolution geometry", fn);
        return 1;
    }
    if (g.H >= HW_LIMIT || g.W >= HW_LIMIT || g.Hk >= HW_LIMIT || g.Wk >= HW_LIMIT) {
        set_error("%s: spatial extent above %d is not supported", fn, HW_LIMIT);
        return 1;
    }
    return 0;
}

static ConvTileDesc forward_desc(const ConvGeom &g, int ns) {
    ConvTileDesc d = {};
    d.in_hwc = g.hwc ? 1 : 0;
    d.batch = ns; d.Cin = g.Ci; d.Hin = g.H; d.Win = g.W;
    d.Cout = g.Co; d.Ho = g.Ho; d.Wo = g.Wo;
    d.KH = g.Hk; d.KW = g.Wk; d.sh = g.sh; d.sw = g.sw;
    d.padU = g.Up; d.padD = g.Dp; d.padL = g.Lp; d.padR = g.Rp;
    d.x_sb = (long long)g.Ci * g.H * g.W; d.x_sc = (long long)g.H * g.W; d.x_sy = g.W;
    return d;
}

// Whether the products with patch matrices (ptl_conv_any.hip) go before the kernels for small problems (raw tiles of one
// image, the gathering product).
// Forward: always.  Over 2800 layers (1 to 250 samples) the other routes take 1.05 to 1.25 times as long in the mean of each
// group of type, layout, stride and bias, and the better one of each layer would give 0 to 4 % more.  Except fp16 layers of
// unit stride with few filters over many pixels and a short contraction, where the raw tiles read each input once: 8 ->
// 16 1 x 1, 14.2 us there and 17.5 here; 64 -> 16 3 x 3, 42 and 49; but 83 -> 16 1 x 1 24 and 16, 132 -> 15 3 x 3 152 and 129.
// And channel-major fp16 layers of several taps without a bias whose few tiles have a long contraction, which takes its partial
// sums through memory here: 58 layers of more than 32 filters, 550 terms and up to 30 tiles of 64 x 64 0.88 of the time by
// the gathering product in the mean, 1.02 at worst (2 samples, 64 -> 152, 13 x 13, 5 x 5 12.6 and 15.2 us; 4, 64 -> 128, 12 x 12,
// 3 x 3 10.7 and 12.1); above 33 tiles 1.00, below 550 terms 1.10, up to 32 filters 0.99, with a bias 1.04.
// One gradient alone: by the millions of multiplications of a step, counted by how full its tiles are.  Strides: the
// other route of the input gradient runs over a zero-stuffed tensor.  A bias gradient is a launch of its own on the other
// routes.  Both routes were timed on 5000 layers (1 to 128 samples, 3 to 512 channels on 7 to 64 pixels, 1 to 25
// taps, strides 1 and 2, tensors in turn), forced one after the other.  Time of the other route over this one's, mean of
// the layers between a third of the line and the line; between the line and three times it; and what the rule loses to the
// better of the two for each layer, in the mean:
//   weight gradient 300: 0.96, 1.07, 4 %; strided 200: 1.00, 1.05, 7 %; channel-minor fp16 20: 1.16, 1.20, 7 %, fp32 300:
//                   1.02, 1.15, 8 %
//   input gradient  strided 15: 1.22, 1.40, 7 %; fp16 300: 0.93, 1.17, 4 %, channel-minor 240: 0.89, 1.13, 3 %; fp32 320:
//                   0.90, 1.11, 4 %, channel-minor 1500: 1.15, 1.16, 4 %; few pixels under many filters, whose re-laying
//                   takes longer than the product, are left out: 0.70
// Where a line lies higher than these figures ask for, layers keep the route they had.
template <typename T>
static bool any_pays(const ConvGeom &g, int ns, int steps, bool bias) {
    if (state().gemm_path >= 7) return true;
    if (state().gemm_path != 0) return false;
    constexpr int VEC = 16 / (int)sizeof(T);
    auto fill = [](double n, int unit) { return n / ((long long)((n + unit - 1) / unit) * unit); };
    const int K = g.Ci * g.Hk * g.Wk;
    const bool strided = g.sh > 1 || g.sw > 1, half = sizeof(T) == 2;
    if (steps == 1) {
        const long long pix = (long long)ns * g.Ho * g.Wo, tiles = (g.Co + 63) / 64 * ((pix + 63) / 64);
        if (half && !g.hwc && !bias && K > g.Ci && K >= 550 && g.Co > 32 && tiles <= 30) return false;
        return !(half && !g.hwc && !strided && g.Co <= 16 && K <= (K == g.Ci ? 40 : 700) && pix > 100000);
    }
    double mflop = 2e-6 * ns * g.Co * g.Ho * g.Wo * K * fill(g.Co, 32) * fill(K, 64);
    if (g.hwc) mflop *= fill(g.Ci, VEC);
    if (bias) mflop *= 1.5;
    if (steps == 2) return mflop >= (g.hwc ? (half ? 20 : 300) : strided ? 200 : 300);
    if ((long long)ns * g.H * g.W < 256 && (long long)g.Co * K > (1 << 18)) return false;
    return mflop >= (strided ? 15 : half ? (g.hwc ? 240 : 300) : g.hwc ? 1500 : 320);
}

// Patch axis over output pixels (sample, ho, wo) and over kernel taps.
static AxisMap pix_axis(const ConvGeom &g, int ns) {
    AxisMap a = {};
    a.n = ns * g.Ho * g.Wo;
    a.d1 = g.Ho;
    a.d0 = g.Wo;
    if (!g.hwc) {
        a.o2 = g.Ci * g.H * g.W;
        a.o1 = g.sh * g.W;
        a.o0 = g.sw;
        a.ob = -g.Up * g.W - g.Lp;
    } else {
        a.o2 = g.H * g.W * g.Ci;
        a.o1 = g.sh * g.W * g.Ci;
        a.o0 = g.sw * g.Ci;
        a.ob = (-g.Up * g.W - g.Lp) * g.Ci;
    }
    a.h1 = g.sh;
    a.hb = -g.Up;
    a.w0 = g.sw;
    a.wb = -g.Lp;
    return a;
}

static AxisMap tap_axis(const ConvGeom &g) {
    AxisMap a = {};
    a.n = g.Ci * g.Hk * g.Wk;
    if (!g.hwc) {  // (ci, hk, wk)
        a.d1 = g.Hk;
        a.d0 = g.Wk;
        a.o2 = g.H * g.W;
        a.o1 = g.W;
        a.o0 = 1;
        a.h1 = 1;
        a.w0 = 1;
    } else {  // (hk, wk, ci)
        a.d1 = g.Wk;
        a.d0 = g.Ci;
        a.o2 = g.W * g.Ci;
        a.o1 = g.Ci;
        a.o0 = 1;
        a.h2 = 1;
        a.w1 = 1;
    }
    return a;
}

// The product behind a step of a pointwise layer; element (co, ci) of the weights lies at co * w_co + ci * w_ci.
static GemmArgs pw_product(int step, const void *X, const void *Wt, const void *dY, void *out, int ns, int Ci, int Co, int HW, bool hwc, int w_co,
                           int w_ci) {
    GemmArgs q = {};
    q.a.HL = q.a.WL = q.b.HL = q.b.WL = 1;
    const int BP = ns * HW;
    if (step == STEP_FW) {
        q.C = out;
        q.K = Ci;
        if (!hwc) {
            q.A = Wt;
            q.B = X;
            q.N = Co;
            q.M = BP;
            q.a.row = axis_plain(Co, Ci);
            q.a.k = axis_plain(Ci, 1);
            q.b.row = axis_two(BP, HW, Ci * HW, 1);
            q.b.k = axis_plain(Ci, HW);
            q.c.n = axis_plain(Co, HW);
            q.c.m = axis_two(BP, HW, Co * HW, 1);
        } else {
            q.A = X;
            q.B = Wt;
            q.N = BP;
            q.M = Co;
            q.a.row = axis_plain(BP, Ci);
            q.a.k = axis_plain(Ci, 1);
            q.b.row = axis_plain(Co, w_co);
            q.b.k = axis_plain(Ci, w_ci);
            q.c.n = axis_plain(BP, Co);
            q.c.m = axis_plain(Co, 1);
        }
    } else if (step == STEP_WGT_GRAD) {
        q.A = dY;
        q.B = X;
        q.C = out;
        q.N = Co;
        q.M = Ci;
        q.K = BP;
        if (!hwc) {
            q.a.row = axis_plain(Co, HW);
            q.a.k = axis_two(BP, HW, Co * HW, 1);
            q.b.row = axis_plain(Ci, HW);
            q.b.k = axis_two(BP, HW, Ci * HW, 1);
        } else {
            q.a.row = axis_plain(Co, 1);
            q.a.k = axis_plain(BP, Co);
            q.b.row = axis_plain(Ci, 1);
            q.b.k = axis_plain(BP, Ci);
        }
        q.c.n = axis_plain(Co, w_co);
        q.c.m = axis_plain(Ci, w_ci);
    } else {
        q.C = out;
        q.K = Co;
        if (!hwc) {
            q.A = Wt;
            q.B = dY;
            q.N = Ci;
            q.M = BP;
            q.a.row = axis_plain(Ci, w_ci);
            q.a.k = axis_plain(Co, w_co);
            q.b.row = axis_two(BP, HW, Co * HW, 1);
            q.b.k = axis_plain(Co, HW);
            q.c.n = axis_plain(Ci, HW);
            q.c.m = axis_two(BP, HW, Ci * HW, 1);
        } else {
            q.A = dY;
            q.B = Wt;
            q.N = BP;
            q.M = Ci;
            q.a.row = axis_plain(BP, Co);
            q.a.k = axis_plain(Co, 1);
            q.b.row = axis_plain(Ci, w_ci);
            q.b.k = axis_plain(Co, w_co);
            q.c.n = axis_plain(BP, Ci);
            q.c.m = axis_plain(Ci, 1);
        }
    }
    return q;
}

// Weight and input gradient (and the bias gradient, where db is not null) of a dense layer over ns samples.  apart: what is
// written shares no memory with what is read.
template <typename T>
static int dense_bw(const T *X, const T *Wt, const T *dY, T *dW, T *dX, T *db, int ns, int in, int out, bool apart) {
    GemmArgs q = {}, r = {};
    q.A = dY;  // dW[o][i] = sum_b dY[b][o] * X[b][i]
    q.B = X;
    q.C = dW;
    q.N = out;
    q.M = in;
    q.K = ns;
    q.a.row = axis_plain(out, 1);
    q.a.k = axis_plain(ns, out);
    q.b.row = axis_plain(in, 1);
    q.b.k = axis_plain(ns, in);
    q.a.HL = q.a.WL = q.b.HL = q.b.WL = 1;
    q.c.n = axis_plain(out, in);
    q.c.m = axis_plain(in, 1);
    r.A = dY;  // dX[b][i] = sum_o dY[b][o] * W[o][i]
    r.B = Wt;
    r.C = dX;
    r.N = ns;
    r.M = in;
    r.K = out;
    r.a.row = axis_plain(ns, out);
    r.a.k = axis_plain(out, 1);
    r.b.row = axis_plain(in, 1);
    r.b.k = axis_plain(out, in);
    r.a.HL = r.a.WL = r.b.HL = r.b.WL = 1;
    r.c.n = axis_plain(ns, in);
    r.c.m = axis_plain(in, 1);
    // Whole slabs of aligned rows: the look-up-free pair.  Other layers, and small ones with a bias (whose gradient
    // would be a launch of its own: 2.5-4 us against the 1-2 us that the pair is faster), take the kernel for any
    // size up to the work at which the look-up-free kernels' larger tiles make up for two launches.
    const double flops = 4.0 * ns * in * out;
    int rc = -1;
    if (!apart) {
        rc = ns == 1 ? mm_dispatch<T>(dY, X, dW, out, in, 1, 0) : gemm<T>(q);
        if (rc == 0 && db) rc = bias_grad<T>(dY, db, ns, out, 1, 1);
        return rc ? rc : mm_dispatch<T>(dY, Wt, dX, ns, in, out, 0);
    }
    if (!db || flops > 4e9) rc = gemm_pair_lean<T>(q, r);
    if (rc < 0 && state().gemm_path == 0 && flops <= (sizeof(T) == 2 ? 3e10 : 1e10)) {
        rc = linear_bw_ragged<T>(X, Wt, dY, dW, dX, db, ns, in, out);
        if (rc >= 0) return rc;
    }
    if (rc < 0) rc = gemm_pair<T>(q, r);
    if (rc == 0 && db) rc = bias_grad<T>(dY, db, ns, out, 1, 1);
    return rc;
}

// Layers of one tap, unit stride and no padding are products of matrices: channel-minor ones dense layers over the pixels.
static bool is_point(const ConvGeom &g) {
    return g.Hk == 1 && g.Wk == 1 && g.sh == 1 && g.sw == 1 && g.H == g.Ho && g.W == g.Wo && g.Up == 0 && g.Lp == 0 && state().gemm_path == 0;
}
// Where the other routes are ahead (over 1800 fp32 and 900 fp16 layers; elsewhere they take 1.2 to 1.3 times as long in the mean):
//   * fp32, channel-major, from 1 GFLOP on: 33 to 128 channels into 256 and more, whose panels of filters each stream the image again
//     (their time over this one's 0.72 to 0.88 in the mean; 128 -> 335, 103 samples of 36 x 25 119 and 241 us); more channels into at
//     most 32, whose tiles are half empty (0.88); and from 2 GFLOP on images of up to 1024 pixels, with which the tiles end (0.94).
//     Images of at most 48 pixels whatever the work from two tiles a compute unit on (0.43 to 0.86; 128 -> 448, 203 samples of 5 x 3
//     15 and 61; one tile 1.0);
//   * fp32, channel-minor, eight to sixteen channels in whole pieces, no bias: the gathering product, which reads each pixel once (8 ->
//     16, 436 samples of 59 x 59 37.5 and 132, 16 -> 320, 98 000 pixels 48.1 and 50.6; 20 -> 184 14.5 and 14.6);
//   * fp16, channel-minor with a bias, at most 32 filters over 2^17 pixels and more, 0.79: the patch products (32 -> 24, 1.7 million
//     pixels 95 and 128; 33 filters and more 1.1).
template <typename T>
static bool point_shallow(const ConvGeom &g, bool bias) {
    return sizeof(T) == 4 && g.hwc && !bias && g.Ci >= 8 && g.Ci <= 16 && g.Ci % 4 == 0 && g.Co % 4 == 0 && is_point(g);
}
template <typename T>
static bool point_fw_behind(const ConvGeom &g, int ns, bool bias) {
    const int P = g.H * g.W;
    if (sizeof(T) == 2) return g.hwc && bias && g.Co <= 32 && (long long)ns * P >= 1 << 17;
    if (g.hwc) return point_shallow<T>(g, bias);
    const double gflop = 2e-9 * ns * P * g.Ci * g.Co;
    if (P <= 48 && (long long)ns * ((g.Co + 63) / 64) >= 2 * state().num_cu) return true;
    return gflop >= 1 && g.Ci > 32 && (g.Ci <= 128 ? g.Co >= 256 : g.Co <= 32 || (P <= 1024 && gflop >= 2));
}
template <typename T>
static int point_fw(const ConvGeom &g, int ns, const T *X, const T *Wt, const T *bias, T *Y) {
    constexpr int VEC = 16 / (int)sizeof(T);
    const int P = g.H * g.W;
    if (!is_point(g) || g.Ci < VEC || P < VEC || point_fw_behind<T>(g, ns, bias != nullptr)) return -1;
    // (fp32 on the kernel for any size: its sums are nearer to 64 bits, 1.1e-7 against 2.0e-7 for 448 -> 47 channels)
    if (sizeof(T) == 4 || (bias && !g.hwc)) return conv_point_fw<T>(forward_desc(g, ns), X, Wt, bias, Y);
    if (g.hwc) return mm_dispatch<T>(X, Wt, Y, ns * P, g.Co, g.Ci, 1, bias);
    return gemm<T>(pw_product(STEP_FW, X, Wt, nullptr, Y, ns, g.Ci, g.Co, P, false, g.Ci, 1));
}
// fp32 layers of 128 channels and more into fewer than 64, from 64 MB of input and output on: half of a tile of the weight gradient
// is empty, and the patch products (channel-major: 0.63 to 0.93 of the time here) or the steps one after the other (channel-minor: 0.67
// to 0.93) are ahead (480 -> 9, 257 samples of 27 x 27 272 and 422 us; 704 -> 16, 12 of 93 x 65 140 and 199; 64 filters 1.0 to 1.2).
template <typename T>
static bool point_bw_behind(const ConvGeom &g, double mb) { return sizeof(T) == 4 && mb >= 64 && g.Co < 64 && g.Ci >= 128; }
// Channel-major tensors: both gradients in one launch, fp16 up to 40 MB of input and output, the two products by themselves
// above (the patch matrices' time over theirs, mean of 400 layers, one launch / two products: fp16 2.4 / 1.6 below 0.3 MB,
// 1.8 / 1.4 at 3 to 30, 1.5 / 1.4 at 30 to 100, 0.8 / 1.2 above).  Channel-minor fp16 layers above 100 MB stay with the
// patch matrices (0.82).
template <typename T>
static int point_bw(const ConvGeom &g, int ns, const T *X, const T *dY, const T *Wt, T *dW, T *dX, T *db) {
    constexpr int VEC = 16 / (int)sizeof(T);
    const int P = g.H * g.W;
    if (!is_point(g) || g.Ci < VEC || g.Co < VEC) return -1;
    const double mb = 1e-6 * sizeof(T) * ns * P * ((double)g.Ci + g.Co);
    if (point_bw_behind<T>(g, mb)) return -1;
    if (g.hwc) {
        if (sizeof(T) == 4) return linear_bw_ragged<T>(X, Wt, dY, dW, dX, db, ns * P, g.Ci, g.Co);
        return mb > 100 ? -1 : dense_bw<T>(X, Wt, dY, dW, dX, db, ns * P, g.Ci, g.Co, true);
    }
    if (P < VEC) return -1;
    if (mb <= 40 || sizeof(T) == 4) {
        const int rc = conv_point_bw<T>(forward_desc(g, ns), X, dY, Wt, dW, dX, db);
        if (rc >= 0) return rc;
    }
    int rc = gemm<T>(pw_product(STEP_WGT_GRAD, X, nullptr, dY, dW, ns, g.Ci, g.Co, P, false, g.Ci, 1));
    if (rc == 0 && db) rc = bias_grad<T>(dY, db, ns, g.Co, P, 0);
    return rc ? rc : gemm<T>(pw_product(STEP_IN_GRAD, nullptr, Wt, dY, dX, ns, g.Ci, g.Co, P, false, g.Ci, 1));
}

template <typename T, typename Args>
static int conv2d_fw(const Args *a, int ns, const char *fn) {
    ConvGeom g;
    if (int rc = conv_geom(a, g, fn, true)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    const int K = g.Ci * g.Hk * g.Wk, P = g.Ho * g.Wo;
    size_t in_n = (size_t)ns * g.Ci * g.H * g.W, out_n = (size_t)ns * g.Co * P;
    if (!fits_int(in_n) || !fits_int(out_n)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    Stager sg;
    const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), in_n);
    const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)g.Co * K);
    T *Y = sg.out(reinterpret_cast<T *>(a->output->data), out_n);
    const T *bias = nullptr;
    if (a->USE_BIASES == 1) {
        if (!a->bias) {
            set_error("%s: USE_BIASES=1 with a null bias blob", fn);
            return 1;
        }
        bias = sg.in(reinterpret_cast<const T *>(a->bias->data), (size_t)g.Co);
    }
    if (sg.failed()) return 2;

    int rc = -1;
    state().last_conv_direct = 0;
    state().last_conv_resident = 0;
    if (state().gemm_path != 1) {
        ConvTileDesc d = forward_desc(g, ns);
        OutMap c;
        if (!g.hwc) {
            d.w_base = 0; d.w_sm = K; d.w_sc = g.Hk * g.Wk; d.w_sy = g.Wk; d.w_sx = 1;
            c.n = axis_two(ns * P, P, g.Co * P, 1);
            c.m = axis_plain(g.Co, P);
        } else {  // X[b][h][w][ci], W[co][hk][wk][ci], Y[b][pix][co]
            d.w_base = 0; d.w_sm = K; d.w_sc = 1; d.w_sy = g.Wk * g.Ci; d.w_sx = g.Ci;
            c.n = axis_plain(ns * P, g.Co);
            c.m = axis_plain(g.Co, 1);
        }
        if (state().gemm_path >= 7 && (rc = conv_any_fw<T>(d, X, Wt, bias, Y)) >= 0) return sg.finish(rc);
        // (the small-layer kernel adds no bias, which is a launch of its own: 8 -> 16 channels on 8 x 8, 7 samples, fp16 8.3
        // against 7.3 us, 8 -> 48 on 40 x 40, 8 samples, fp32 17.5 against 8.4; without one its bits are those of the call
        // that also forms the output's sums)
        if (bias && !conv_small_pre_pending() && (rc = point_fw<T>(g, ns, X, Wt, bias, Y)) >= 0) return sg.finish(rc);
        if (bias && !conv_small_pre_pending() && any_pays<T>(g, ns, 1, true) && (rc = conv_any_fw<T>(d, X, Wt, bias, Y)) >= 0) return sg.finish(rc);
        if (!g.hwc) rc = conv_small<T>(d, X, Wt, Y);
        // (a normalisation to apply on the way in is the small-layer kernel's business alone: nothing was launched)
        if (rc == CONV_PRE_REFUSED || conv_small_pre_pending()) return CONV_PRE_REFUSED;
        if (rc < 0 && (rc = point_fw<T>(g, ns, X, Wt, bias, Y)) >= 0) return sg.finish(rc);
        // Large fp32 layers are bound by the matrix instructions, of which products with patch matrices form theirs from bf16
        // pieces: from 3 GFLOP on 1.2 to 1.7 times as fast as tap by tap, 0.96 at worst (60 samples, 128 -> 128, 32 x 32, 3 x 3 175
        // -> 139 us; 4, 512 -> 64, 28 x 28, 5 x 5 channel-minor 145 -> 85), 0.75 to 1.26 from 1 to 2.5 GFLOP.
        const bool gather = point_shallow<T>(g, bias != nullptr);
        if (rc < 0 && !gather && sizeof(T) == 4 && state().gemm_path == 0 && 2.0 * ns * g.Co * g.Ho * g.Wo * K >= 3e9 &&
            any_pays<T>(g, ns, 1, bias != nullptr) && (rc = conv_any_fw<T>(d, X, Wt, bias, Y)) >= 0)
            return sg.finish(rc);
        if (rc < 0) rc = conv_taps<T>(d, X, Wt, Y, c);
        if (rc < 0 && !gather && any_pays<T>(g, ns, 1, bias != nullptr) && (rc = conv_any_fw<T>(d, X, Wt, bias, Y)) >= 0) return sg.finish(rc);
        if (rc < 0) rc = conv_tile<T>(d, X, Wt, Y, c);
        if (rc > 0) return sg.finish(rc);
        if (rc == 0) state().last_conv_direct = 1;
    }
    GemmArgs q = {};
    q.K = K;
    OperandMap wmap = {}, pmap = {};
    wmap.row = axis_plain(g.Co, K);
    wmap.k = axis_plain(K, 1);
    wmap.HL = wmap.WL = 1;
    pmap.row = pix_axis(g, ns);
    pmap.k = tap_axis(g);
    pmap.HL = g.H;
    pmap.WL = g.W;
    if (!g.hwc) {  // Y[b][co][pix]
        q.A = Wt;
        q.B = X;
        q.N = g.Co;
        q.M = ns * P;
        q.a = wmap;
        q.b = pmap;
        q.c.n = axis_plain(g.Co, P);
        q.c.m = axis_two(q.M, P, g.Co * P, 1);
    } else {  // Y[b][pix][co]
        q.A = X;
        q.B = Wt;
        q.N = ns * P;
        q.M = g.Co;
        q.a = pmap;
        q.b = wmap;
        q.c.n = axis_plain(q.N, g.Co);
        q.c.m = axis_plain(g.Co, 1);
    }
    q.C = Y;
    if (rc < 0) rc = gemm<T>(q);
    if (rc == 0 && bias) {
        launch_bias_add<T>(Y, bias, out_n, g.Co, g.hwc ? 1 : P);
        if (!hip_ok(hipGetLastError(), "bias add launch")) rc = 2;
    }
    return sg.finish(rc);
}

template <typename T, typename Args>
static int conv2d_wg(const Args *a, int ns, const char *fn) {
    ConvGeom g;
    if (int rc = conv_geom(a, g, fn, true)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    const int K = g.Ci * g.Hk * g.Wk, P = g.Ho * g.Wo;
    size_t in_n = (size_t)ns * g.Ci * g.H * g.W, out_n = (size_t)ns * g.Co * P;
    if (!fits_int(in_n) || !fits_int(out_n)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    Stager sg;
    const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), in_n);
    const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), out_n);
    T *dW = sg.out(reinterpret_cast<T *>(a->coeff->diff), (size_t)g.Co * K);
    T *db = nullptr;
    if (a->USE_BIASES == 1) {
        if (!a->bias) {
            set_error("%s: USE_BIASES=1 with a null bias blob", fn);
            return 1;
        }
        db = sg.out(reinterpret_cast<T *>(a->bias->diff), (size_t)g.Co);
    }
    if (sg.failed()) return 2;

    int rc = -1;
    state().last_conv_direct = 0;
    state().last_conv_resident = 0;
    if (state().gemm_path != 1) {
        const ConvTileDesc d = forward_desc(g, ns);
        // the kernel with resident channel-blocked tiles where it is preferred; else the resident output tile kernel,
        // else (or on request) the sum over taps.  From 256 channels on either side and 16384 output pixels the sum
        // over taps goes before the output tile kernel (measured: 81 against 91 us for 256 -> 256 on 14x14 at batch
        // 128, 455 against 533 us on 28x28 at batch 256; at batch 8 the output tile kernel takes 26 against 34 us)
        if (state().gemm_path >= 7 && (rc = conv_any_bw<T>(d, X, dY, nullptr, dW, nullptr, db)) >= 0) return sg.finish(rc);
        const bool taps_first = d.Cin >= 128 && d.Cout >= 128 && (d.Cin >= 256 || d.Cout >= 256) &&
                                (long long)ns * g.Ho * g.Wo >= 16384;
        if (g.hwc) {  // channel-minor tensors: the sum over taps from 64 channels on, else the gathering GEMM below
            if (!any_pays<T>(g, ns, 2, db != nullptr) || (sizeof(T) == 2 && conv_halo_wg_hwc_fits(d, X, dY) && conv_halo_wg_hwc_preferred(d)))
                rc = conv_taps_wg<T>(d, X, dY, dW);
        } else if ((rc = conv_small_wg<T>(d, X, dY, dW,
                                           static_cast<const void *>(dW) == static_cast<const void *>(a->coeff->diff))) >= 0) {
            // (small 3x3 layers: one launch for the partial sums over sample ranges, one to add them)
        } else {
            const bool tiles_resident = sizeof(T) == 2 && state().gemm_path == 0 && conv_halo_wg_preferred(d);
            if (state().gemm_path == 3 || state().gemm_path == 5 || tiles_resident || (taps_first && state().gemm_path != 2))
                rc = conv_taps_wg<T>(d, X, dY, dW);
            if (rc < 0) rc = conv_tile_wg<T>(d, X, dY, dW);
            if (rc < 0 && state().gemm_path != 3) rc = conv_taps_wg<T>(d, X, dY, dW);
        }
        if (rc < 0 && any_pays<T>(g, ns, 2, db != nullptr) && (rc = conv_any_bw<T>(d, X, dY, nullptr, dW, nullptr, db)) >= 0) return sg.finish(rc);
        if (rc > 0) return sg.finish(rc);
        if (rc == 0) state().last_conv_direct = 1;
    }
    GemmArgs q = {};
    q.A = dY;
    q.B = X;
    q.C = dW;
    q.N = g.Co;
    q.M = K;
    q.K = ns * P;
    if (!g.hwc) {
        q.a.row = axis_plain(g.Co, P);
        q.a.k = axis_two(q.K, P, g.Co * P, 1);
    } else {
        q.a.row = axis_plain(g.Co, 1);
        q.a.k = axis_plain(q.K, g.Co);
    }
    q.a.HL = q.a.WL = 1;
    q.b.row = tap_axis(g);
    q.b.k = pix_axis(g, ns);
    q.b.HL = g.H;
    q.b.WL = g.W;
    q.c.n = axis_plain(g.Co, K);
    q.c.m = axis_plain(K, 1);
    if (rc < 0) rc = gemm<T>(q);
    if (rc == 0 && db) rc = bias_grad<T>(dY, db, ns, g.Co, P, g.hwc);
    return sg.finish(rc);
}

template <typename T, typename Args>
static int conv2d_ig(const Args *a, int ns, const char *fn) {
    ConvGeom g;
    if (int rc = conv_geom(a, g, fn, false)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    const int Pk = g.Hk * g.Wk, K = g.Co * Pk, P = g.Ho * g.Wo;
    size_t in_n = (size_t)ns * g.Ci * g.H * g.W, out_n = (size_t)ns * g.Co * P;
    const int Hd = (g.Ho - 1) * g.sh + 1, Wd = (g.Wo - 1) * g.sw + 1;
    size_t dil_n = (size_t)ns * g.Co * Hd * Wd;
    if (!fits_int(in_n) || !fits_int(out_n) || !fits_int(dil_n)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    Stager sg;
    const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)g.Co * g.Ci * Pk);
    const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), out_n);
    T *dX = sg.out(reinterpret_cast<T *>(a->input->diff), in_n);
    if (sg.failed()) return 2;

    // A strided single-tap layer without padding (projection shortcut): only the input positions the layer read
    // get a gradient, dX[ci][sh*u][sw*v] = sum_co W[co][ci] dY[co][u][v] - one plain product written through a
    // strided output map into the zeroed tensor (the general route below would run a stride-1 pass over a
    // zero-stuffed gradient four times the size: measured 32 against 11 us for 16 -> 32 channels, 32x32, batch 128).
    // With bottom / right padding the last output rows or columns sit on padded positions outside the input;
    // the scatter map has no coordinate test, so such geometries take the general route below.
    const bool taps_inside = (long long)(g.Ho - 1) * g.sh < g.H && (long long)(g.Wo - 1) * g.sw < g.W;
    if (Pk == 1 && (g.sh != 1 || g.sw != 1) && g.Up == 0 && g.Lp == 0 && taps_inside && state().gemm_path != 1) {
        const int vec = reinterpret_cast<uintptr_t>(dX) % 16 == 0;
        const size_t threads = vec ? (in_n + 16 / sizeof(T) - 1) / (16 / sizeof(T)) : in_n;
        hipLaunchKernelGGL((zero_kernel<T>), dim3(blocks_for(threads)), dim3(256), 0, state().stream, dX, in_n, vec);
        if (!hip_ok(hipGetLastError(), "zero launch")) return sg.finish(2);
        state().last_conv_direct = 0;
        GemmArgs q = {};
        q.K = g.Co;
        q.C = dX;
        q.a.HL = q.a.WL = q.b.HL = q.b.WL = 1;
        AxisMap pix = {};  // output pixel (sample, u, v) inside the input tensor
        pix.n = ns * P;
        pix.d1 = g.Ho;
        pix.d0 = g.Wo;
        if (!g.hwc) {
            q.A = Wt;
            q.B = dY;
            q.N = g.Ci;
            q.M = ns * P;
            q.a.row = axis_plain(g.Ci, 1);
            q.a.k = axis_plain(g.Co, g.Ci);
            q.b.row = axis_two(q.M, P, g.Co * P, 1);
            q.b.k = axis_plain(g.Co, P);
            pix.o2 = g.Ci * g.H * g.W;
            pix.o1 = g.sh * g.W;
            pix.o0 = g.sw;
            q.c.n = axis_plain(g.Ci, g.H * g.W);
            q.c.m = pix;
        } else {
            q.A = dY;
            q.B = Wt;
            q.N = ns * P;
            q.M = g.Ci;
            q.a.row = axis_plain(q.N, g.Co);
            q.a.k = axis_plain(g.Co, 1);
            q.b.row = axis_plain(g.Ci, 1);
            q.b.k = axis_plain(g.Co, g.Ci);
            pix.o2 = g.H * g.W * g.Ci;
            pix.o1 = g.sh * g.W * g.Ci;
            pix.o0 = g.sw * g.Ci;
            q.c.n = pix;
            q.c.m = axis_plain(g.Ci, 1);
        }
        return sg.finish(gemm<T>(q));
    }

    if (state().gemm_path >= 7) {
        ConvTileDesc d = {};
        d.in_hwc = g.hwc ? 1 : 0;
        d.batch = ns; d.Cin = g.Ci; d.Hin = g.H; d.Win = g.W;
        d.Cout = g.Co; d.Ho = g.Ho; d.Wo = g.Wo;
        d.KH = g.Hk; d.KW = g.Wk; d.sh = g.sh; d.sw = g.sw;
        d.padU = g.Up; d.padD = g.Dp; d.padL = g.Lp; d.padR = g.Rp;
        const int rc = conv_any_bw<T>(d, nullptr, dY, Wt, nullptr, dX, nullptr);
        if (rc >= 0) return sg.finish(rc);
    }
    // Small stride-2 layers (3x3 or 1x1): the small-layer kernel stuffs the zeros while it fills its LDS tile.
    if (!g.hwc && g.sh == 2 && g.sw == 2 && g.Hk == g.Wk && (g.Hk == 3 || g.Hk == 1)) {
        ConvTileDesc d = {};
        d.batch = ns; d.Cin = g.Co; d.Hin = g.Ho; d.Win = g.Wo; d.in_dil = 2;
        d.Cout = g.Ci; d.Ho = g.H; d.Wo = g.W;
        d.KH = g.Hk; d.KW = g.Wk; d.sh = 1; d.sw = 1;
        d.padU = g.Hk - 1 - g.Up; d.padL = g.Wk - 1 - g.Lp;
        d.padD = g.H + g.Hk - 1 - Hd - d.padU; d.padR = g.W + g.Wk - 1 - Wd - d.padL;
        d.x_sb = (long long)g.Co * P; d.x_sc = P; d.x_sy = g.Wo;
        d.w_base = Pk - 1; d.w_sm = Pk; d.w_sc = g.Ci * Pk; d.w_sy = -g.Wk; d.w_sx = -1;
        state().last_conv_direct = 0;
        state().last_conv_resident = 0;
        const int rc = conv_small<T>(d, dY, Wt, dX);
        if (rc == 0) state().last_conv_direct = 1;
        if (rc >= 0) return sg.finish(rc);
    }

    if ((g.sh != 1 || g.sw != 1) && any_pays<T>(g, ns, 4, false)) {
        const int rc = conv_any_bw<T>(forward_desc(g, ns), nullptr, dY, Wt, nullptr, dX, nullptr);
        if (rc >= 0) return sg.finish(rc);
    }

    // A strided forward is undone by a unit-stride pass over the zero-stuffed gradient.
    if (g.sh != 1 || g.sw != 1) {
        T *dil = static_cast<T *>(scratch(dil_n * sizeof(T)));
        if (!dil) return 2;
        hipLaunchKernelGGL((dilate_kernel<T>), dim3((unsigned)(g.hwc ? ns : ns * g.Co)), dim3(256), 0, state().stream, dY,
                           dil, g.Ho, g.Wo, Hd, Wd, g.sh, g.sw, g.hwc ? g.Co : 1);
        if (!hip_ok(hipGetLastError(), "dilate launch")) return sg.finish(2);
        dY = dil;
    }

    // dX[ci,hi,wi] = sum_{co,hk,wk} W[co,ci,hk,wk] * dYd[co, hi+Up-hk, wi+Lp-wk]
    OperandMap wmap = {}, gmap = {};
    wmap.HL = wmap.WL = 1;
    gmap.HL = Hd;
    gmap.WL = Wd;
    gmap.row.n = ns * g.H * g.W;
    gmap.row.d1 = g.H;
    gmap.row.d0 = g.W;
    gmap.row.h1 = 1;
    gmap.row.hb = g.Up;
    gmap.row.w0 = 1;
    gmap.row.wb = g.Lp;
    gmap.k.n = K;
    state().last_conv_direct = 0;
    state().last_conv_resident = 0;
    if (state().gemm_path != 1) {
        ConvTileDesc d = {};
        d.batch = ns; d.Cin = g.Co; d.Hin = Hd; d.Win = Wd;
        d.Cout = g.Ci; d.Ho = g.H; d.Wo = g.W;
        d.KH = g.Hk; d.KW = g.Wk; d.sh = 1; d.sw = 1;
        d.padU = g.Hk - 1 - g.Up; d.padL = g.Wk - 1 - g.Lp;
        d.padD = g.H + g.Hk - 1 - Hd - d.padU; d.padR = g.W + g.Wk - 1 - Wd - d.padL;
        d.x_sb = (long long)g.Co * Hd * Wd; d.x_sc = (long long)Hd * Wd; d.x_sy = Wd;
        OutMap c;
        if (!g.hwc) {
            d.w_base = Pk - 1; d.w_sm = Pk; d.w_sc = g.Ci * Pk; d.w_sy = -g.Wk; d.w_sx = -1;
            c.n = axis_two(ns * g.H * g.W, g.H * g.W, g.Ci * g.H * g.W, 1);
            c.m = axis_plain(g.Ci, g.H * g.W);
        } else {  // dY[b][pix][co], W[co][hk][wk][ci], dX[b][pix][ci]
            d.in_hwc = 1;
            d.w_base = (Pk - 1) * g.Ci; d.w_sm = 1; d.w_sc = Pk * g.Ci; d.w_sy = -g.Wk * g.Ci; d.w_sx = -g.Ci;
            c.n = axis_plain(ns * g.H * g.W, g.Ci);
            c.m = axis_plain(g.Ci, 1);
        }
        // (the zero-stuffed gradient of a strided layer lives in the scratch buffer the tap route would reuse)
        int rc = !g.hwc ? conv_small<T>(d, dY, Wt, dX) : -1;
        if (rc < 0 && g.sh == 1 && g.sw == 1) rc = conv_taps<T>(d, dY, Wt, dX, c);
        if (rc < 0 && g.sh == 1 && g.sw == 1 && any_pays<T>(g, ns, 4, false) &&
            (rc = conv_any_bw<T>(forward_desc(g, ns), nullptr, dY, Wt, nullptr, dX, nullptr)) >= 0)
            return sg.finish(rc);
        if (rc < 0) rc = conv_tile<T>(d, dY, Wt, dX, c);
        if (rc == 0) state().last_conv_direct = 1;
        if (rc >= 0) return sg.finish(rc);
    }
    GemmArgs q = {};
    q.K = K;
    q.C = dX;
    if (!g.hwc) {
        wmap.row = axis_plain(g.Ci, Pk);
        wmap.k = axis_two(K, Pk, g.Ci * Pk, 1);  // (co, tap)
        gmap.row.o2 = g.Co * Hd * Wd;
        gmap.row.o1 = Wd;
        gmap.row.o0 = 1;
        gmap.row.ob = g.Up * Wd + g.Lp;
        gmap.k.d1 = g.Hk;  // (co, hk, wk)
        gmap.k.d0 = g.Wk;
        gmap.k.o2 = Hd * Wd;
        gmap.k.o1 = -Wd;
        gmap.k.o0 = -1;
        gmap.k.h1 = -1;
        gmap.k.w0 = -1;
        q.A = Wt;
        q.B = dY;
        q.N = g.Ci;
        q.M = ns * g.H * g.W;
        q.a = wmap;
        q.b = gmap;
        q.c.n = axis_plain(g.Ci, g.H * g.W);
        q.c.m = axis_two(q.M, g.H * g.W, g.Ci * g.H * g.W, 1);
    } else {
        // contraction index (hk, wk, co); weights are [co][hk][wk][ci]
        wmap.row = axis_plain(g.Ci, 1);
        wmap.k.n = K;
        wmap.k.d1 = g.Wk;
        wmap.k.d0 = g.Co;
        wmap.k.o2 = g.Wk * g.Ci;
        wmap.k.o1 = g.Ci;
        wmap.k.o0 = Pk * g.Ci;
        gmap.row.o2 = Hd * Wd * g.Co;
        gmap.row.o1 = Wd * g.Co;
        gmap.row.o0 = g.Co;
        gmap.row.ob = (g.Up * Wd + g.Lp) * g.Co;
        gmap.k.d1 = g.Wk;
        gmap.k.d0 = g.Co;
        gmap.k.o2 = -Wd * g.Co;
        gmap.k.o1 = -g.Co;
        gmap.k.o0 = 1;
        gmap.k.h2 = -1;
        gmap.k.w1 = -1;
        q.A = dY;
        q.B = Wt;
        q.N = ns * g.H * g.W;
        q.M = g.Ci;
        q.a = gmap;
        q.b = wmap;
        q.c.n = axis_plain(q.N, g.Ci);
        q.c.m = axis_plain(g.Ci, 1);
    }
    return sg.finish(gemm<T>(q));
}

// ---- Pointwise convolution ------------------------------------------------------------
// CHW: X[b][Ci][HW], W[Co][Ci], Y[b][Co][HW].
// HWC: X[b][HW][Ci], Y[b][HW][Co]; weights are [Ci][Co] in the fp32 layer
// (lib/sources/pulp_conv_pw_fp32.c:67-74) and [Co][Ci] in the fp16 layer
// (lib/sources/pulp_conv_pw_fp16.c:70-76).

template <typename Args>
static int pw_geom(const Args *a, const char *fn) {
    if (!a || !a->input || !a->coeff || !a->output) {
        printf("[%s] null argument structure\n", fn);
        set_error("%s: null argument structure", fn);
        return 1;
    }
    if (a->HWC != 0 && a->HWC != 1) {
        printf("[%s] Invalid HWC parameter!\n", fn);
        set_error("%s: HWC must be 0 or 1", fn);
        return 1;
    }
    if (a->input->C <= 0 || a->output->C <= 0 || a->input->H <= 0 || a->input->W <= 0 ||
        a->input->H != a->output->H || a->input->W != a->output->W) {
        printf("[%s] invalid tensor geometry\n", fn);
        set_error("%s: invalid tensor geometry", fn);
        return 1;
    }
    return 0;
}

// Weight and input gradient of one call (the batched twin of pulp_conv2d_*_bw_cl): honours skip_wg_grad /
// skip_in_grad; where both run on the resident-tile kernels they share the blocked copy of the output gradient.
template <typename T, typename Args>
static int conv2d_bw_routes(const Args *a, int ns, const char *fn) {
    const bool wg = a->skip_wg_grad == 0, ig = a->skip_in_grad == 0;
    bool apart = false;
    if (wg && ig && ns >= 1 && a->input && a->coeff && a->output) {
        auto at = [](const void *p) { return static_cast<const T *>(p); };
        auto n = [&](const auto *b) { return (size_t)ns * (size_t)std::max(b->C, 0) * std::max(b->H, 0) * std::max(b->W, 0); };
        const size_t nw = (size_t)std::max(a->output->C, 0) * std::max(a->input->C, 0) * std::max(a->coeff->H, 0) * std::max(a->coeff->W, 0);
        apart = !backward_shares_memory<T>(at(a->input->data), n(a->input), at(a->coeff->data), nw, at(a->output->diff), n(a->output),
                                           at(a->coeff->diff), at(a->input->diff),
                                           a->USE_BIASES == 1 && a->bias ? at(a->bias->diff) : nullptr, (size_t)std::max(a->output->C, 0));
    }
    state().last_gemm_form = 0;
    if (apart && a->USE_BIASES != 1) {
        ConvGeom g;
        if (int rc = conv_geom(a, g, fn, true)) return rc;
        const int P = g.Ho * g.Wo, Pk = g.Hk * g.Wk, K = g.Ci * Pk;
        size_t in_n = (size_t)ns * g.Ci * g.H * g.W, out_n = (size_t)ns * g.Co * P;
        const bool unit = g.sh == 1 && g.sw == 1 && g.Up + g.Dp == g.Hk - 1 && g.Lp + g.Rp == g.Wk - 1;
        const bool halving = g.sh == 2 && g.sw == 2;  // (small layers only: the zeros are stuffed on the way into LDS)
        if (!g.hwc && g.Hk == g.Wk && (g.Hk == 3 || g.Hk == 1) && (unit || halving) && fits_int(in_n) && fits_int(out_n) &&
            (state().gemm_path == 0 || state().gemm_path == 5 || state().gemm_path == 6)) {
            if (!ensure_init()) return 2;
            ConvTileDesc f = {}, b = {};
            f.batch = ns; f.Cin = g.Ci; f.Hin = g.H; f.Win = g.W;
            f.Cout = g.Co; f.Ho = g.Ho; f.Wo = g.Wo;
            f.KH = g.Hk; f.KW = g.Wk; f.sh = g.sh; f.sw = g.sw;
            f.padU = g.Up; f.padD = g.Dp; f.padL = g.Lp; f.padR = g.Rp;
            f.x_sb = (long long)g.Ci * g.H * g.W; f.x_sc = (long long)g.H * g.W; f.x_sy = g.W;
            // the input gradient: a unit-stride pass over the output gradient, zero-stuffed where the forward strode
            const int Hd = (g.Ho - 1) * g.sh + 1, Wd = (g.Wo - 1) * g.sw + 1;
            b.batch = ns; b.Cin = g.Co; b.Hin = g.Ho; b.Win = g.Wo; b.in_dil = halving ? 2 : 0;
            b.Cout = g.Ci; b.Ho = g.H; b.Wo = g.W;
            b.KH = g.Hk; b.KW = g.Wk; b.sh = 1; b.sw = 1;
            b.padU = g.Hk - 1 - g.Up; b.padL = g.Wk - 1 - g.Lp;
            b.padD = g.H + g.Hk - 1 - Hd - b.padU; b.padR = g.W + g.Wk - 1 - Wd - b.padL;
            b.x_sb = (long long)g.Co * P; b.x_sc = P; b.x_sy = g.Wo;
            b.w_base = Pk - 1; b.w_sm = Pk; b.w_sc = g.Ci * Pk; b.w_sy = -g.Wk; b.w_sx = -1;
            // small layers: both products in one launch; wide layers: one shared copy of the output gradient
            const bool small = g.Ci <= 64 && g.Co <= 64 && g.W % (16 / (int)sizeof(T)) == 0 && state().gemm_path != 5;
            const bool wide = unit && g.Hk == 3 && sizeof(T) == 2 && ns > 1 && state().gemm_path != 6 && conv_halo_wg_preferred(f);
            if (small || wide) {
                Stager sg;
                const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), in_n);
                const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), out_n);
                const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)g.Co * K);
                T *dW = sg.out(reinterpret_cast<T *>(a->coeff->diff), (size_t)g.Co * K);
                T *dX = sg.out(reinterpret_cast<T *>(a->input->diff), in_n);
                if (sg.failed()) return sg.rejected() ? 1 : 2;
                state().last_conv_direct = 0;
                state().last_conv_resident = 0;
                // (a host tensor's gradient is a staging copy that this call copies back: its sums cannot wait)
                const bool on_device = static_cast<const void *>(dW) == static_cast<const void *>(a->coeff->diff);
                int rc = small ? conv_small_bw<T>(f, b, X, dY, Wt, dW, dX, on_device) : -1;
                if (rc < 0 && wide) rc = conv_halo_bw<T>(f, b, X, dY, Wt, dW, dX);
                if (rc >= 0) {
                    if (rc == 0) state().last_conv_direct = 1;
                    return sg.finish(rc);
                }
                // neither kernel took the layer: nothing was written, so nothing of the staged gradients goes back
                // to the caller; the two single-step calls below are the only writers
                sg.discard();
            }
        }
    }
    // Both gradients as products with patch matrices (small and middling layers: in one launch), whatever the size: over 2300
    // layers of 1 to 250 samples the other routes take 1.2 to 1.7 times as long in the mean of each group of type, layout,
    // stride and bias, and taking the better one of each layer would give 1 % more.  Except where one of the gradients
    // has a kernel of its own that is ahead: the raw-tile weight gradient of unit-stride 3x3 layers from 10 GFLOP on (other over
    // this: 1.18 in the mean at 3 to 6 GFLOP, 1.06 at 6 to 10, 0.98 at 10 to 20, 0.94 above; 1x1 layers 1.2 above 10), the
    // resident-tile one wherever it is preferred (a call then has the bits of its two steps), and those of channel-minor
    // layers from 20 on (1.77, 1.26 and 1.22 at 4, 10 and 19, 0.92 and 0.82 at 31 and 39).  Strided channel-major 1x1 layers,
    // whose input gradient is a plain product scattered over zeros, from some MB of input and output on (fp16 1.4 in the
    // mean at 3 to 5 MB, 1.0 at 7 to 30, 0.8 above; fp32 1.4 at 7 to 10, 1.1 at 10 to 30, 0.8 above).  Channel-minor ones of whole
    // groups of 32 filters, for the same reason: fp16 from 32768 output pixels on (0.73 to 0.99 of the time here in the mean; 40 -> 64, 196
    // samples of 109 x 75 81 and 192 us), fp32 without a bias from 32 MB on with at most 32 channels on one side (0.87 and 0.94; more 1.07).
    // And fp16 layers of up to sixteen channels on rows of whole pieces, from 60000 pixels on, whose gradients both have kernels on raw
    // tiles (6 -> 8, 449 samples of 40 x 40 58 and 107, 9 -> 7, 29 of 160 x 112 64 and 100, 11 -> 4, 4 of 160 x 160 36 and 36).
    if (apart && (a->USE_BIASES != 1 || a->bias)) {
        ConvGeom g;
        if (int rc = conv_geom(a, g, fn, true)) return rc;
        if (!ensure_init()) return 2;
        const int P = g.Ho * g.Wo, K = g.Ci * g.Hk * g.Wk;
        const size_t in_n = (size_t)ns * g.Ci * g.H * g.W, out_n = (size_t)ns * g.Co * P;
        const ConvTileDesc d = forward_desc(g, ns);
        const double gflop = 2e-9 * ns * g.Co * P * K;
        const bool own_wg = g.sh == 1 && g.sw == 1 && sizeof(T) == 2 && !g.hwc && K > g.Ci && g.Hk <= 3 &&
                            (gflop >= 10 || (g.Hk == 3 && g.Wk == 3 && conv_halo_wg_preferred(d)));
        const bool resident = sizeof(T) == 2 && g.hwc && gflop >= 20 && conv_halo_wg_hwc_fits(d, nullptr, nullptr) && conv_halo_wg_hwc_preferred(d);
        const bool scatter = K == g.Ci && (g.sh > 1 || g.sw > 1) && !g.hwc && sizeof(T) * (in_n + out_n) >= (sizeof(T) == 2 ? 7000000 : 30000000);
        const bool forced = state().gemm_path >= 7, bias = a->USE_BIASES == 1;
        const double mb = 1e-6 * sizeof(T) * (in_n + out_n);
        const bool point_steps = is_point(g) && g.hwc && point_bw_behind<T>(g, mb);
        const bool minor_steps = g.hwc && K == g.Ci && (g.sh > 1 || g.sw > 1) && g.Co % 32 == 0 &&
                                 (sizeof(T) == 2 ? (long long)ns * P >= 32768 : !bias && mb >= 32 && std::min(g.Ci, g.Co) <= 32);
        const bool small_steps = sizeof(T) == 2 && !g.hwc && g.Hk == 3 && g.Wk == 3 && g.sh == 1 && g.sw == 1 && g.W % 8 == 0 && g.Ci <= 16 &&
                                 g.Co <= 16 && (long long)ns * P >= 60000;
        const bool steps = own_wg || resident || scatter || point_steps || minor_steps || small_steps;
        if ((forced || (state().gemm_path == 0 && !steps)) && fits_int(in_n) && fits_int(out_n)) {
            Stager sg;
            const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), in_n);
            const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), out_n);
            const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)g.Co * K);
            T *dW = sg.out(reinterpret_cast<T *>(a->coeff->diff), (size_t)g.Co * K);
            T *dX = sg.out(reinterpret_cast<T *>(a->input->diff), in_n);
            T *db = a->USE_BIASES == 1 ? sg.out(reinterpret_cast<T *>(a->bias->diff), (size_t)g.Co) : nullptr;
            if (sg.failed()) return sg.rejected() ? 1 : 2;
            state().last_conv_direct = 0;
            state().last_conv_resident = 0;
            int rc = point_bw<T>(g, ns, X, dY, Wt, dW, dX, db);
            if (rc < 0) rc = conv_any_bw<T>(d, X, dY, Wt, dW, dX, db);
            if (rc >= 0) return sg.finish(rc);
            sg.discard();
        }
    }
    const int rc = wg ? conv2d_wg<T>(a, ns, fn) : 0;
    return rc == 0 && ig ? conv2d_ig<T>(a, ns, fn) : rc;
}

template <typename T, typename Args>
static int conv2d_bw(const Args *a, int ns, const char *fn) {
    if (!a) {
        set_error("%s: null argument structure", fn);
        return 1;
    }
    ptl_internal_stage_begin();  // (host tensors: fetched once for both steps, and for a route that was asked before them)
    return ptl_internal_stage_end(conv2d_bw_routes<T>(a, ns, fn));
}

template <typename T, typename Args>
static int pw_step(const Args *a, int ns, int step, const char *fn) {
    if (int rc = pw_geom(a, fn)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    const int Ci = a->input->C, Co = a->output->C, HW = a->input->H * a->input->W;
    const bool hwc = a->HWC == 1;
    const bool w_ci_major = hwc && sizeof(T) == 4;  // fp32 HWC stores [Ci][Co]
    const int w_co = w_ci_major ? 1 : Ci, w_ci = w_ci_major ? Co : 1;
    size_t in_n = (size_t)ns * Ci * HW, out_n = (size_t)ns * Co * HW;
    if (!fits_int(in_n) || !fits_int(out_n)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    Stager sg;
    const size_t w_n = (size_t)Co * Ci;
    const T *X = step != STEP_IN_GRAD ? sg.in(reinterpret_cast<const T *>(a->input->data), in_n) : nullptr;
    const T *dY = step != STEP_FW ? sg.in(reinterpret_cast<const T *>(a->output->diff), out_n) : nullptr;
    const T *Wt = step != STEP_WGT_GRAD ? sg.in(reinterpret_cast<const T *>(a->coeff->data), w_n) : nullptr;
    T *out = step == STEP_FW ? sg.out(reinterpret_cast<T *>(a->output->data), out_n)
             : step == STEP_WGT_GRAD ? sg.out(reinterpret_cast<T *>(a->coeff->diff), w_n)
                                     : sg.out(reinterpret_cast<T *>(a->input->diff), in_n);
    const GemmArgs q = pw_product(step, X, Wt, dY, out, ns, Ci, Co, HW, hwc, w_co, w_ci);
    if (sg.failed()) return 2;
    return sg.finish(gemm<T>(q));
}

// ---- Linear --------------------------------------------------------------------------
// W is [out][in] row-major (lib/sources/pulp_linear_fp32.c:39-46); sample b of
// the input/output blobs is a vector of blob->dim elements.

// Few samples: the kernels of ptl_gemm.hip that read each weight once, against tiles of 32 x 32 and more with partial sums, in a
// grid of 64 to 65536 inputs and 64 to 65536 outputs.  Other routes' time over theirs:
// Forward, up to sixteen samples: 1.1 to 2.2 while the weights are few.  Every row reads all samples again, 4 to 16 times the
// weights' own bytes out of L2, which bounds it beyond
//   two samples        nothing (8192 x 8192 fp32 1.13, fp16 1.11)
//   three and four     70 MB (64 MB: fp32 1.07 to 1.24, fp16 0.97 to 1.13; 128 MB: 0.83 to 1.07)
//   five to eight      24 MB of rows up to 16384 (16 MB: 1.08 to 1.36; 32 MB: 0.62 to 1.0; 65536 -> 64 0.78 and 0.96)
//   up to sixteen      5.5 MB of rows up to 12 KB and 4096, 1280 outputs (5 MB: 1.01 to 1.12; 10 MB and 4096 -> 320: 0.7 to 0.9)
// and rows by the thousand, of which each is a wave's chain of shuffles: 8192 of less than 1 KB take 0.75 to 0.92, 65536 of any
// length 0.2 to 0.8, 16384 0.5 to 0.9 but with two samples from 4 KB on (1.1 to 2.0) and in fp32 with up to four from 2 KB on,
// where the other routes are behind up to 256 MB (1.3 to 1.75).
template <typename T>
static bool few_fw(int ns, int in, int out) {
    if (state().gemm_path != 0 || ns < 2 || ns > 16) return false;
    const double bytes = (double)sizeof(T) * in * out, row = (double)sizeof(T) * in;
    if (ns > 8) return out <= 1280 && in <= 4096 && row <= 12288 && bytes <= 5.5e6;
    const bool more = out > 8192;
    if (more && !(ns == 2 && row >= 4096) && !(sizeof(T) == 4 && ns <= 4 && out <= 16384 && row >= 2048)) return false;
    if (out > 4096 && row < 1024) return false;
    if (ns > 4) return in <= 16384 && bytes <= 24e6;
    return ns == 2 || bytes <= (more ? 270e6 : 70e6);
}
// Backward: fp32 1.0 to 3.7 (2304 -> 2100, 4 samples 45 -> 11 us; 4096 -> 64 0.85 to 0.93), fp16 1.0 to 2.7 up to four samples.  With
// more the matrix instructions of fp16 are as fast until the weights are many (8 samples, 640 -> 48 5.1 and 5.7 us, 1157 -> 500
// 7.9 -> 7.3, 640 -> 2100 12.3 -> 10.1), and with one side long and the other short (65536 -> 64 0.74, 16384 -> 64 0.83, 64 ->
// 65536 0.9; 8192 -> 64 1.02, 64 -> 16384 1.08).
template <typename T>
static bool few_bw(int ns, int in, int out) {
    if (state().gemm_path != 0 || ns < 2 || ns > LINEAR_FEW) return false;
    return sizeof(T) == 4 || ns <= 4 || ((in >= 1024 || out >= 1536) && in <= 128LL * out && out <= 512LL * in);
}

template <typename T, typename Args>
static int linear_step(const Args *a, int ns, int step, const char *fn) {
    if (!a || !a->input || !a->coeff || !a->output) {
        printf("[%s] null argument structure\n", fn);
        set_error("%s: null argument structure", fn);
        return 1;
    }
    const int in = a->input->dim, out = a->output->dim;
    if (in <= 0 || out <= 0) {
        printf("[%s] invalid tensor geometry\n", fn);
        set_error("%s: invalid tensor geometry", fn);
        return 1;
    }
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    if (!fits_int((size_t)ns * in) || !fits_int((size_t)ns * out) || !fits_int((size_t)in * out)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    const bool use_bias = a->use_biases == 1;
    if (use_bias && !a->bias) {
        set_error("%s: use_biases=1 with a null bias blob", fn);
        return 1;
    }
    Stager sg;
    int rc = 0;
    if (step == STEP_FW) {
        const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), (size_t)ns * in);
        const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)out * in);
        T *Y = sg.out(reinterpret_cast<T *>(a->output->data), (size_t)ns * out);
        const T *bias = use_bias ? sg.in(reinterpret_cast<const T *>(a->bias->data), (size_t)out) : nullptr;
        if (sg.failed()) return 2;
        if (few_fw<T>(ns, in, out)) return sg.finish(linear_few_fw<T>(X, Wt, Y, bias, ns, in, out));
        rc = mm_dispatch<T>(X, Wt, Y, ns, out, in, 1, bias);  // Y[b][o] = X[b][:] . W[o][:] + bias[o]
    } else if (step == STEP_BW_BOTH) {
        // weight and input gradient of a batch in one launch
        const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), (size_t)ns * in);
        const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)out * in);
        const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), (size_t)ns * out);
        T *dW = sg.out(reinterpret_cast<T *>(a->coeff->diff), (size_t)out * in);
        T *dX = sg.out(reinterpret_cast<T *>(a->input->diff), (size_t)ns * in);
        T *db = use_bias ? sg.out(reinterpret_cast<T *>(a->bias->diff), (size_t)out) : nullptr;
        if (sg.failed()) return 2;
        const bool apart = !backward_shares_memory<T>(X, (size_t)ns * in, Wt, (size_t)out * in, dY, (size_t)ns * out, dW, dX, db, (size_t)out);
        if (few_bw<T>(ns, in, out) && apart) return sg.finish(linear_few_bw<T>(X, Wt, dY, dW, dX, db, ns, in, out));
        if (ns == 1 && apart) return sg.finish(linear_one_bw<T>(X, Wt, dY, dW, dX, db, in, out));
        rc = dense_bw<T>(X, Wt, dY, dW, dX, db, ns, in, out, apart);
    } else if (step == STEP_WGT_GRAD) {
        const T *X = sg.in(reinterpret_cast<const T *>(a->input->data), (size_t)ns * in);
        const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), (size_t)ns * out);
        T *dW = sg.out(reinterpret_cast<T *>(a->coeff->diff), (size_t)out * in);
        T *db = use_bias ? sg.out(reinterpret_cast<T *>(a->bias->diff), (size_t)out) : nullptr;
        if (sg.failed()) return 2;
        if (ns == 1) {
            rc = mm_dispatch<T>(dY, X, dW, out, in, 1, 0);
        } else {  // dW[o][i] = sum_b dY[b][o] * X[b][i]
            GemmArgs q = {};
            q.A = dY;
            q.B = X;
            q.C = dW;
            q.N = out;
            q.M = in;
            q.K = ns;
            q.a.row = axis_plain(out, 1);
            q.a.k = axis_plain(ns, out);
            q.b.row = axis_plain(in, 1);
            q.b.k = axis_plain(ns, in);
            q.a.HL = q.a.WL = q.b.HL = q.b.WL = 1;
            q.c.n = axis_plain(out, in);
            q.c.m = axis_plain(in, 1);
            rc = gemm<T>(q);
        }
        if (rc == 0 && db) rc = bias_grad<T>(dY, db, ns, out, 1, 1);  // db[o] = sum_b dY[b][o]
    } else {
        const T *Wt = sg.in(reinterpret_cast<const T *>(a->coeff->data), (size_t)out * in);
        const T *dY = sg.in(reinterpret_cast<const T *>(a->output->diff), (size_t)ns * out);
        T *dX = sg.out(reinterpret_cast<T *>(a->input->diff), (size_t)ns * in);
        if (sg.failed()) return 2;
        rc = mm_dispatch<T>(dY, Wt, dX, ns, in, out, 0);  // dX[b][i] = sum_o dY[b][o] * W[o][i]
    }
    return sg.finish(rc);
}

template <typename T>
static int bias_add_mat(T *mat, const T *bias, int N, int M, int per_row) {
    if (N <= 0 || M <= 0) return 0;
    if (!mat || !bias) {
        set_error("bias add: null argument");
        return 1;
    }
    if (!ensure_init()) return 2;
    Stager sg;
    size_t total = (size_t)N * M;
    T *m = sg.inout(mat, total);
    const T *b = sg.in(bias, (size_t)(per_row ? N : M));
    if (sg.failed()) return 2;
    launch_bias_add<T>(m, b, total, per_row ? N : M, per_row ? M : 1);
    return sg.finish(hip_ok(hipGetLastError(), "bias add launch") ? 0 : 2);
}

template <typename T>
static int rowsum_mat(const T *mat, T *out, int N, int K) {
    if (N <= 0 || K <= 0) return 0;
    if (!mat || !out) {
        set_error("row sum: null argument");
        return 1;
    }
    if (!ensure_init()) return 2;
    Stager sg;
    const T *m = sg.in(mat, (size_t)N * K);
    T *o = sg.out(out, (size_t)N);
    if (sg.failed()) return 2;
    return sg.finish(bias_grad<T>(m, o, 1, N, K, 0));
}

template <typename T, typename Args>
static int conv2d_fw_stats(const Args *a, int ns, ::ptl_norm_stats *st, const char *fn) {
    if (!st) {
        set_error("%s: null statistics struct", fn);
        return 1;
    }
    st->valid = 0;
    const bool take = a && a->USE_BIASES != 1;  // (a bias is added by a launch behind the kernel that forms the sums)
    if (take) conv_small_stats_to(st);
    const int rc = conv2d_fw<T>(a, ns, fn);
    conv_small_stats_to(nullptr);
    if (rc) st->valid = 0;
    return rc;
}

// The forward call of a normalisation layer and of the convolution that reads its output, in that order - as one
// launch where the small-layer kernel takes the convolution (it then applies the normalisation to its input tile while
// it loads it and writes the normalisation's output on the way), as the two calls otherwise.  Same results bit for bit.
template <typename T, typename Args, typename NormArgs, typename Fusion>
static int conv2d_fw_normed(const Args *a, int ns, ::ptl_norm_stats *st_out, const NormArgs *n, const Fusion *f,
                            const ::ptl_norm_stats *st_in, int (*norm_call)(const NormArgs *, const Fusion *,
                                                                            const ::ptl_norm_stats *),
                            const char *fn) {
    if (!a || !n) {
        set_error("%s: null argument", fn);
        return 1;
    }
    if (st_out) st_out->valid = 0;
    const bool shapes = a->input && n->input && n->output && n->output->data && n->output->data == a->input->data &&
                        n->input->data && n->weight_data && n->bias_data && n->eps && ns > 0 && n->B == ns &&
                        n->C == a->input->C && n->H == a->input->H && n->W == a->input->W && n->C > 0 && n->H > 0 && n->W > 0;
    const bool sums = st_in && st_in->valid == 1 && st_in->part && st_in->parts > 0 && shapes && st_in->channels == n->C &&
                      st_in->count == (size_t)ns * n->H * n->W &&
                      (size_t)n->C * st_in->parts * 4 * sizeof(float) <= st_in->bytes;
    if (sums && ensure_init() && state().gemm_path != 1) {
        const size_t cnt = (size_t)ns * n->C * n->H * n->W;
        bool device;
        {
            Stager sg(true);  // (host tensors: the two calls, which stage them)
            (void)sg.in(reinterpret_cast<const T *>(n->input->data), cnt);
            (void)sg.out(reinterpret_cast<T *>(n->output->data), cnt);
            if (f && f->skip) (void)sg.in(reinterpret_cast<const T *>(f->skip), cnt);
            (void)sg.in(reinterpret_cast<const T *>(n->weight_data), (size_t)n->C);
            (void)sg.in(reinterpret_cast<const T *>(n->bias_data), (size_t)n->C);
            (void)sg.in(reinterpret_cast<const T *>(n->eps), (size_t)1);
            device = !sg.failed();
        }
        if (device) {
            ConvPreNorm pre = {};
            pre.x = n->input->data;
            pre.out = n->output->data;
            pre.skip = f ? f->skip : nullptr;
            pre.weight = n->weight_data;
            pre.bias = n->bias_data;
            pre.eps = n->eps;
            pre.part = st_in->part;
            pre.parts = st_in->parts;
            pre.relu = f && f->relu ? 1 : 0;
            pre.count = st_in->count;
            conv_small_pre_to(&pre);
            const int rc = st_out ? conv2d_fw_stats<T>(a, ns, st_out, fn) : conv2d_fw<T>(a, ns, fn);
            conv_small_pre_to(nullptr);
            if (rc != CONV_PRE_REFUSED) return rc;
        }
    }
    if (int rc = norm_call(n, f, st_in)) return rc;
    return st_out ? conv2d_fw_stats<T>(a, ns, st_out, fn) : conv2d_fw<T>(a, ns, fn);
}

// Backward step whose input gradient becomes the gradient a normalisation in front of this layer starts from:
// input->diff = (dX [+ post->add]) [where post->mask > 0, else 0], rounded to T after the sum like a tensor an
// element-wise layer would have written, and the sums of that gradient and of its products with post->x in `sums`
// (valid = 1) - when the small-layer kernel takes the layer.  Any other route leaves the plain input gradient and
// sums->valid = 0.  Device tensors only.
template <typename T, typename Args>
static int conv2d_bw_post(const Args *a, int ns, ::ptl_wg_batch *batch, const ::ptl_grad_post *post,
                          ::ptl_norm_stats *sums, const char *fn) {
    if (!post || !sums || !post->x) {
        set_error("%s: null gradient epilogue or statistics struct", fn);
        return 1;
    }
    sums->valid = 0;
    if (!a || !a->input || !a->input->diff || a->skip_in_grad) {
        set_error("%s: the gradient epilogue needs the input gradient", fn);
        return 1;
    }
    if (ns <= 0 || a->input->C <= 0 || a->input->H <= 0 || a->input->W <= 0) {
        set_error("%s: invalid tensor geometry", fn);
        return 1;
    }
    if (!ensure_init()) return 2;
    const size_t n = (size_t)ns * a->input->C * a->input->H * a->input->W;
    {
        Stager sg(true);  // host tensors are rejected
        (void)sg.inout(reinterpret_cast<T *>(a->input->diff), n);
        if (post->add) (void)sg.in(reinterpret_cast<const T *>(post->add), n);
        if (post->mask) (void)sg.in(reinterpret_cast<const T *>(post->mask), n);
        (void)sg.in(reinterpret_cast<const T *>(post->x), n);
        if (sg.failed()) return sg.rejected() ? 1 : 2;
    }
    conv_small_defer_to(batch);
    conv_small_post_to(post, sums);
    const int rc = conv2d_bw<T>(a, ns, fn);
    conv_small_post_to(nullptr, nullptr);
    conv_small_defer_to(nullptr);
    if (rc) sums->valid = 0;
    return rc;
}

}  // namespace ptl

// ---- C ABI -------------------------------------------------------------------------------
using ptl::half_t;

extern "C" {

void ptl_internal_set_status(int s) { ptl::set_status(s); }
int ptl_internal_bias_add_fp32(float *mat, const float *bias, int N, int M, int per_row) {
    return ptl::bias_add_mat<float>(mat, bias, N, M, per_row);
}
int ptl_internal_bias_add_fp16(fp16 *mat, const fp16 *bias, int N, int M, int per_row) {
    return ptl::bias_add_mat<half_t>(reinterpret_cast<half_t *>(mat), reinterpret_cast<const half_t *>(bias), N, M,
                                     per_row);
}
int ptl_internal_rowsum_fp32(const float *mat, float *out, int N, int K) {
    return ptl::rowsum_mat<float>(mat, out, N, K);
}
int ptl_internal_rowsum_fp16(const fp16 *mat, fp16 *out, int N, int K) {
    return ptl::rowsum_mat<half_t>(reinterpret_cast<const half_t *>(mat), reinterpret_cast<half_t *>(out), N, K);
}

int ptl_conv2d_fp32_fw_batched(const struct Conv2D_args *a, int ns) {
    return ptl::conv2d_fw<float>(a, ns, "pulp_conv2d_fp32_fw_cl");
}
int ptl_conv2d_fp32_wg_batched(const struct Conv2D_args *a, int ns) {
    return ptl::conv2d_wg<float>(a, ns, "pulp_conv2d_fp32_bw_param_grads_cl");
}
int ptl_conv2d_fp32_ig_batched(const struct Conv2D_args *a, int ns) {
    return ptl::conv2d_ig<float>(a, ns, "pulp_conv2d_fp32_bw_input_grads_cl");
}
int ptl_conv2d_fp16_fw_batched(const struct Conv2D_args_fp16 *a, int ns) {
    return ptl::conv2d_fw<half_t>(a, ns, "pulp_conv2d_fp16_fw_cl");
}
int ptl_conv2d_fp16_wg_batched(const struct Conv2D_args_fp16 *a, int ns) {
    return ptl::conv2d_wg<half_t>(a, ns, "pulp_conv2d_fp16_bw_param_grads_cl");
}
int ptl_conv2d_fp16_ig_batched(const struct Conv2D_args_fp16 *a, int ns) {
    return ptl::conv2d_ig<half_t>(a, ns, "pulp_conv2d_fp16_bw_input_grads_cl");
}
int ptl_conv2d_fp32_bw_batched(const struct Conv2D_args *a, int ns) {
    return ptl::conv2d_bw<float>(a, ns, "pulp_conv2d_fp32_bw_cl");
}
int ptl_conv2d_fp16_bw_batched(const struct Conv2D_args_fp16 *a, int ns) {
    return ptl::conv2d_bw<half_t>(a, ns, "pulp_conv2d_fp16_bw_cl");
}

size_t ptl_conv2d_fp16_cache_bytes(const struct Conv2D_args_fp16 *a, int ns) {
    ptl::ConvGeom g;
    if (ns <= 0 || ptl::conv_geom(a, g, "ptl_conv2d_fp16_cache_bytes", false)) return 0;
    if (g.hwc || g.Hk != 3 || g.Wk != 3 || g.sh != 1 || g.sw != 1 || g.Ci % 64 != 0) return 0;
    ptl::ConvTileDesc d = {};
    d.batch = ns; d.Cin = g.Ci; d.Hin = g.H; d.Win = g.W;
    d.Cout = g.Co; d.Ho = g.Ho; d.Wo = g.Wo;
    d.KH = 3; d.KW = 3; d.sh = 1; d.sw = 1;
    d.padU = g.Up; d.padD = g.Dp; d.padL = g.Lp; d.padR = g.Rp;
    int Hp, Wp;
    ptl::conv_padded_grid(d, &Hp, &Wp);
    if (!ptl::conv_halo_fits(d, Hp, Wp)) return 0;
    return ((size_t)(g.Ci / 8) * ns * Hp * Wp + (size_t)ptl::conv_halo_margin()) * 16;
}
int ptl_conv2d_fp16_fw_batched_cached(const struct Conv2D_args_fp16 *a, int ns, struct ptl_conv_cache *c) {
    if (c) c->valid = 0;
    ptl::conv_cache_set(c, nullptr);
    const int rc = ptl::conv2d_fw<half_t>(a, ns, "pulp_conv2d_fp16_fw_cl");
    ptl::conv_cache_set(nullptr, nullptr);
    return rc;
}
int ptl_conv2d_fp16_cache_prepare(const struct Conv2D_args_fp16 *reader, int ns, struct ptl_conv_cache *c) {
    if (!c) {
        ptl::set_error("ptl_conv2d_fp16_cache_prepare: no cache");
        return 1;
    }
    c->valid = 0;
    const size_t need = ptl_conv2d_fp16_cache_bytes(reader, ns);
    ptl::ConvGeom g;
    if (need == 0 || ptl::conv_geom(reader, g, "ptl_conv2d_fp16_cache_prepare", false)) {
        ptl::set_error("ptl_conv2d_fp16_cache_prepare: the layer does not read a blocked copy of its input");
        return 1;
    }
    if (!c->buf || c->bytes < need || reinterpret_cast<uintptr_t>(c->buf) % 16 != 0) {
        ptl::set_error("ptl_conv2d_fp16_cache_prepare: the buffer must be 16-byte aligned device memory of %zu bytes", need);
        return 1;
    }
    if (!ptl::ensure_init()) return 2;
    // zero halo, zero margin: the producing layer only ever writes the pixels
    const size_t n = need / 2;  // halves, 8 per thread
    hipLaunchKernelGGL((ptl::zero_kernel<half_t>), dim3(ptl::blocks_for((n + 7) / 8)), dim3(256), 0, ptl::state().stream,
                       static_cast<half_t *>(c->buf), n, 8);
    if (!ptl::hip_ok(hipGetLastError(), "zero launch")) return 2;
    ptl::ConvTileDesc d = {};
    d.Hin = g.H; d.Win = g.W; d.padU = g.Up; d.padD = g.Dp; d.padL = g.Lp; d.padR = g.Rp;
    int Hp, Wp;
    ptl::conv_padded_grid(d, &Hp, &Wp);
    const int geo[6] = {ns, g.Ci, Hp, Wp, g.Up, g.Lp};
    for (int i = 0; i < 6; ++i) c->geometry[i] = geo[i];
    return 0;
}
int ptl_conv2d_fp16_fw_batched_chained(const struct Conv2D_args_fp16 *a, int ns, struct ptl_conv_cache *in,
                                       struct ptl_conv_cache *out) {
    if (out) out->valid = 0;
    // (a bias is added by a launch behind the convolution kernel: the copy would miss it, so none is written)
    if (a && a->USE_BIASES == 1) out = nullptr;
    const bool have = in && in->valid;
    ptl::conv_cache_set(have ? nullptr : in, nullptr);
    ptl::conv_cache_chain(have ? in : nullptr, out);
    const int rc = ptl::conv2d_fw<half_t>(a, ns, "pulp_conv2d_fp16_fw_cl");
    ptl::conv_cache_set(nullptr, nullptr);
    ptl::conv_cache_chain(nullptr, nullptr);
    return rc;
}
int ptl_conv2d_fp16_wg_batched_cached(const struct Conv2D_args_fp16 *a, int ns, const struct ptl_conv_cache *c) {
    ptl::conv_cache_set(nullptr, c);
    const int rc = ptl::conv2d_wg<half_t>(a, ns, "pulp_conv2d_fp16_bw_param_grads_cl");
    ptl::conv_cache_set(nullptr, nullptr);
    return rc;
}
int ptl_conv2d_fp16_bw_batched_cached(const struct Conv2D_args_fp16 *a, int ns, const struct ptl_conv_cache *c) {
    ptl::conv_cache_set(nullptr, c);
    const int rc = ptl::conv2d_bw<half_t>(a, ns, "pulp_conv2d_fp16_bw_cl");
    ptl::conv_cache_set(nullptr, nullptr);
    return rc;
}

int ptl_conv2d_fp16_bw_batched_deferred(const struct Conv2D_args_fp16 *a, int ns, struct ptl_wg_batch *batch) {
    ptl::conv_small_defer_to(batch);
    const int rc = ptl::conv2d_bw<half_t>(a, ns, "pulp_conv2d_fp16_bw_cl");
    ptl::conv_small_defer_to(nullptr);
    return rc;
}
int ptl_conv2d_fp32_bw_batched_deferred(const struct Conv2D_args *a, int ns, struct ptl_wg_batch *batch) {
    ptl::conv_small_defer_to(batch);
    const int rc = ptl::conv2d_bw<float>(a, ns, "pulp_conv2d_fp32_bw_cl");
    ptl::conv_small_defer_to(nullptr);
    return rc;
}
int ptl_conv2d_fp16_fw_batched_normed(const struct Conv2D_args_fp16 *a, int ns, struct ptl_norm_stats *st,
                                      const struct BatchNorm_args_fp16 *norm, const struct ptl_norm_fusion_fp16 *f,
                                      const struct ptl_norm_stats *norm_st) {
    return ptl::conv2d_fw_normed<half_t>(a, ns, st, norm, f, norm_st, ptl_batch_norm_fused_fp16_fw_stats,
                                         "pulp_conv2d_fp16_fw_cl");
}
int ptl_conv2d_fp32_fw_batched_normed(const struct Conv2D_args *a, int ns, struct ptl_norm_stats *st,
                                      const struct BatchNorm_args_fp32 *norm, const struct ptl_norm_fusion_fp32 *f,
                                      const struct ptl_norm_stats *norm_st) {
    return ptl::conv2d_fw_normed<float>(a, ns, st, norm, f, norm_st, ptl_batch_norm_fused_fp32_fw_stats,
                                        "pulp_conv2d_fp32_fw_cl");
}
int ptl_conv2d_fp16_bw_batched_deferred_post(const struct Conv2D_args_fp16 *a, int ns, struct ptl_wg_batch *batch,
                                             const struct ptl_grad_post *post, struct ptl_norm_stats *sums) {
    return ptl::conv2d_bw_post<half_t>(a, ns, batch, post, sums, "pulp_conv2d_fp16_bw_cl");
}
int ptl_conv2d_fp32_bw_batched_deferred_post(const struct Conv2D_args *a, int ns, struct ptl_wg_batch *batch,
                                             const struct ptl_grad_post *post, struct ptl_norm_stats *sums) {
    return ptl::conv2d_bw_post<float>(a, ns, batch, post, sums, "pulp_conv2d_fp32_bw_cl");
}
int ptl_conv2d_fp16_fw_batched_stats(const struct Conv2D_args_fp16 *a, int ns, struct ptl_norm_stats *st) {
    return ptl::conv2d_fw_stats<half_t>(a, ns, st, "pulp_conv2d_fp16_fw_cl");
}
int ptl_conv2d_fp32_fw_batched_stats(const struct Conv2D_args *a, int ns, struct ptl_norm_stats *st) {
    return ptl::conv2d_fw_stats<float>(a, ns, st, "pulp_conv2d_fp32_fw_cl");
}
int ptl_conv2d_fp16_wg_flush(struct ptl_wg_batch *batch) { return ptl::conv_small_flush<half_t>(batch); }
int ptl_conv2d_fp32_wg_flush(struct ptl_wg_batch *batch) { return ptl::conv_small_flush<float>(batch); }

int ptl_conv_pw_fp32_fw_batched(const struct PointWise_Conv_args *a, int ns) {
    return ptl::pw_step<float>(a, ns, STEP_FW, "pulp_conv_pw_fp32_fw_cl");
}
int ptl_conv_pw_fp32_wg_batched(const struct PointWise_Conv_args *a, int ns) {
    return ptl::pw_step<float>(a, ns, STEP_WGT_GRAD, "pulp_conv_pw_fp32_bw_param_grads_cl");
}
int ptl_conv_pw_fp32_ig_batched(const struct PointWise_Conv_args *a, int ns) {
    return ptl::pw_step<float>(a, ns, STEP_IN_GRAD, "pulp_conv_pw_fp32_bw_input_grads_cl");
}
int ptl_conv_pw_fp16_fw_batched(const struct PointWise_Conv_args_fp16 *a, int ns) {
    return ptl::pw_step<half_t>(a, ns, STEP_FW, "pulp_conv_pw_fp16_fw_cl");
}
int ptl_conv_pw_fp16_wg_batched(const struct PointWise_Conv_args_fp16 *a, int ns) {
    return ptl::pw_step<half_t>(a, ns, STEP_WGT_GRAD, "pulp_conv_pw_fp16_bw_param_grads_cl");
}
int ptl_conv_pw_fp16_ig_batched(const struct PointWise_Conv_args_fp16 *a, int ns) {
    return ptl::pw_step<half_t>(a, ns, STEP_IN_GRAD, "pulp_conv_pw_fp16_bw_input_grads_cl");
}

int ptl_linear_fp32_fw_batched(const struct Linear_args *a, int ns) {
    return ptl::linear_step<float>(a, ns, STEP_FW, "pulp_linear_fp32_fw_cl");
}
int ptl_linear_fp32_wg_batched(const struct Linear_args *a, int ns) {
    return ptl::linear_step<float>(a, ns, STEP_WGT_GRAD, "pulp_linear_fp32_bw_param_grads_cl");
}
int ptl_linear_fp32_ig_batched(const struct Linear_args *a, int ns) {
    return ptl::linear_step<float>(a, ns, STEP_IN_GRAD, "pulp_linear_fp32_bw_input_grads_cl");
}
int ptl_linear_fp16_fw_batched(const struct Linear_args_fp16 *a, int ns) {
    return ptl::linear_step<half_t>(a, ns, STEP_FW, "pulp_linear_fp16_fw_cl");
}
int ptl_linear_fp16_wg_batched(const struct Linear_args_fp16 *a, int ns) {
    return ptl::linear_step<half_t>(a, ns, STEP_WGT_GRAD, "pulp_linear_fp16_bw_param_grads_cl");
}
int ptl_linear_fp32_bw_batched(const struct Linear_args *a, int ns) {
    if (a && (a->skip_wg_grad || a->skip_in_grad)) {  // one of the two
        int rc = a->skip_wg_grad ? 0 : ptl::linear_step<float>(a, ns, STEP_WGT_GRAD, "pulp_linear_fp32_bw_cl");
        if (rc == 0 && !a->skip_in_grad) rc = ptl::linear_step<float>(a, ns, STEP_IN_GRAD, "pulp_linear_fp32_bw_cl");
        return rc;
    }
    return ptl::linear_step<float>(a, ns, STEP_BW_BOTH, "pulp_linear_fp32_bw_cl");
}
int ptl_linear_fp16_bw_batched(const struct Linear_args_fp16 *a, int ns) {
    if (a && (a->skip_wg_grad || a->skip_in_grad)) {  // one of the two
        int rc = a->skip_wg_grad ? 0 : ptl::linear_step<half_t>(a, ns, STEP_WGT_GRAD, "pulp_linear_fp16_bw_cl");
        if (rc == 0 && !a->skip_in_grad) rc = ptl::linear_step<half_t>(a, ns, STEP_IN_GRAD, "pulp_linear_fp16_bw_cl");
        return rc;
    }
    return ptl::linear_step<half_t>(a, ns, STEP_BW_BOTH, "pulp_linear_fp16_bw_cl");
}
int ptl_linear_fp16_ig_batched(const struct Linear_args_fp16 *a, int ns) {
    return ptl::linear_step<half_t>(a, ns, STEP_IN_GRAD, "pulp_linear_fp16_bw_input_grads_cl");
}

int ptl_mm_fp32(const float *A, const float *B, float *C, int N, int M, int K, int trans_B) {
    if (N < 0 || M < 0 || K < 0 || !A || !B || !C) {
        ptl::set_error("ptl_mm_fp32: invalid arguments");
        return 1;
    }
    if (!ptl::ensure_init()) return 2;
    ptl::Stager sg;
    const float *dA = sg.in(A, (size_t)N * K);
    const float *dB = sg.in(B, (size_t)K * M);
    float *dC = K > 0 ? sg.out(C, (size_t)N * M) : C;
    if (sg.failed()) return 2;
    return sg.finish(ptl::mm_dispatch<float>(dA, dB, dC, N, M, K, trans_B));
}

int ptl_mm_fp16(const fp16 *A, const fp16 *B, fp16 *C, int N, int M, int K, int trans_B) {
    if (N < 0 || M < 0 || K < 0 || !A || !B || !C) {
        ptl::set_error("ptl_mm_fp16: invalid arguments");
        return 1;
    }
    if (!ptl::ensure_init()) return 2;
    ptl::Stager sg;
    const half_t *dA = sg.in(reinterpret_cast<const half_t *>(A), (size_t)N * K);
    const half_t *dB = sg.in(reinterpret_cast<const half_t *>(B), (size_t)K * M);
    half_t *dC = K > 0 ? sg.out(reinterpret_cast<half_t *>(C), (size_t)N * M) : reinterpret_cast<half_t *>(C);
    if (sg.failed()) return 2;
    return sg.finish(ptl::mm_dispatch<half_t>(dA, dB, dC, N, M, K, trans_B));
}

}  // extern "C"
