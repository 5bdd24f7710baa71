// Conv2D layers of any geometry (up to 25 taps, strides up to 2 x 2, any size and alignment) as products with implicit
// patch matrices (ptl_ragged_conv.inc): what the descriptions of their operands say.
//   * backward, small and middling layers: both gradients in one launch and one more for the partial sums of both; the
//     filters are read where they are, or re-laid together with channel-minor copies of the tensors.
//   * forward: one launch.  Weight gradient alone: one launch.  Input gradient: a strided layer's is split into its phases (the
//     pixels that the same taps reach), each a unit-stride product with its share of the taps - a pass over a zero-stuffed
//     gradient has stride^2 times the work - all in one launch.  The filters it reads are re-laid by spare blocks of the
//     weight gradient's launch.
#include "ptl_common.hpp"
#include "ptl_conv_tile.hpp"
#include "ptl_ragged.hpp"

#include <string.h>

namespace ptl {

constexpr unsigned long long RAG_TENSOR_MAX = 0xf0000000ull;  // bytes: offsets have 32 bits and one that is rejected

// The image side of a layer: the tensor that the patches are taken from.
struct AnyImage {
    int C, H, W, hwc;
    long long bytes;
};

// qh x qw pixels, their first at (y0, x0), step (sy, sx), taps th x tw in direction dir.
template <typename T>
static int any_geo(RagGeo &g, RagOp &o, const void *t, const AnyImage &m, int qh, int qw, int y0, int x0, int sy, int sx, int th, int tw, int dir) {
    constexpr long long ES = (long long)sizeof(T);
    constexpr int VEC = 16 / (int)ES;
    const long long chan = m.hwc ? m.C : 1, pixel = chan * ES;  // bytes from pixel to pixel
    g.d_x = rag_div(qw);
    g.d_y = rag_div(qh);
    g.pb = (unsigned)(ES * m.C * m.H * m.W);
    g.py = (unsigned)(sy * m.W * pixel);
    g.px = (unsigned)(sx * pixel);
    g.y0 = y0;
    g.x0 = x0;
    g.sy = sy;
    g.sx = sx;
    g.ty = g.tx = dir;
    g.H = m.H;
    g.W = m.W;
    const int taps = th * tw;
    g.d_t = rag_div(taps);
    g.d_kw = rag_div(tw);
    for (int t = 0; t < taps; t += tw) g.every_row |= 1u << t;
    for (int t = 0; t < 32 && taps > 0; t += m.hwc ? 32 : taps) g.every_channel |= 1u << t;
    g.all_taps = (1u << taps) - 1u;
    const int pieces = (m.C + VEC - 1) / VEC;
    g.d_cb = rag_div(pieces);
    g.cut = (unsigned)((pieces * VEC - m.C) * ES);
    g.plane = (unsigned)(m.hwc ? pixel : ES * m.H * m.W);
    g.zeros = static_cast<const char *>(state().zeros);
    long long at = ((long long)y0 * m.W + x0) * pixel;
    if (!m.hwc) {
        const long long low = dir < 0 && taps > 0 ? ((long long)(th - 1) * m.W + tw - 1) * ES : 0;
        for (int j = 0, jx = 0, jy = 0, c = 0; j < RAG_TAB && taps > 0; ++j) {
            g.tab[j] = (int)((long long)c * g.plane + dir * ((long long)jy * m.W + jx) * ES + low);
            if (++jx == tw) {
                jx = 0;
                if (++jy == th) {
                    jy = 0;
                    ++c;
                }
            }
        }
        at -= low;
        if (m.bytes - at <= 0 || m.bytes - at > (long long)RAG_TENSOR_MAX) return -1;
        g.size = (unsigned)(m.bytes - at);
    }
    o.p = static_cast<const char *>(t) + at;
    return 0;
}

template <typename T>
static RagOp any_rows(const void *p, int rows, long long row_bytes) {  // a matrix contiguous along k
    RagOp o = {};
    o.p = static_cast<const char *>(p);
    o.rows = rows;
    o.row_b = (unsigned)row_bytes;
    return o;
}

static bool any_fits(const ConvTileDesc &d, int es) {
    const long long x = (long long)d.batch * d.Cin * d.Hin * d.Win * es, y = (long long)d.batch * d.Cout * d.Ho * d.Wo * es;
    return d.KH * d.KW <= RAG_TAPS && d.sh <= 2 && d.sw <= 2 && x < (long long)RAG_TENSOR_MAX / 2 && y < (long long)RAG_TENSOR_MAX / 2 &&
           (long long)d.Cout * d.Cin * d.KH * d.KW * es < (1ll << 31) && (long long)d.Cin * d.KH * d.KW * es < (1 << 24) &&
           (long long)d.Cout * d.KH * d.KW * es < (1 << 24) && (long long)d.Ho * d.Wo * es < (1 << 24);
}

static int any_padded(int c, int es) { return (c + 16 / es - 1) / (16 / es) * (16 / es); }  // channels, in whole pieces

// The input pixels sh*u + ph, sw*v + pw: input row sh*u + ph lies under tap ky of output row u + a - jy, ky = k0 + sh*jy.
struct AnyPhase {
    int ph, pw, qh, qw, ky, kx, th, tw, y0, x0;
};
static int any_phases(const ConvTileDesc &d, AnyPhase (&f)[RAG_CONV_MAX]) {
    int n = 0;
    for (int ph = 0; ph < d.sh && ph < d.Hin; ++ph)
        for (int pw = 0; pw < d.sw && pw < d.Win; ++pw) {
            AnyPhase &q = f[n++];
            const int ky = (ph + d.padU) % d.sh, kx = (pw + d.padL) % d.sw;
            q = {ph, pw, (d.Hin - ph + d.sh - 1) / d.sh, (d.Win - pw + d.sw - 1) / d.sw, ky, kx,
                 ky < d.KH ? (d.KH - ky + d.sh - 1) / d.sh : 0, kx < d.KW ? (d.KW - kx + d.sw - 1) / d.sw : 0,
                 (ph + d.padU - ky) / d.sh, (pw + d.padL - kx) / d.sw};
        }
    return n;
}

// Sizes of a step's products.
enum AnyStep { ANY_FW = 1, ANY_WG = 2, ANY_IG = 4 };
template <typename T>
static int any_sizes(const ConvTileDesc &d, int step, bool minor, RagProd (&p)[RAG_CONV_MAX]) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES, SK = 128 / ES;
    const int taps = d.KH * d.KW, P = d.Ho * d.Wo, npix = d.batch * P;
    auto set = [&](RagProd &q, int n, int m, int k) {
        q.N = n;
        q.M = q.m_in = m;
        q.K = k;
        q.runs = q.outer = 1;
    };
    if (step == ANY_WG) {
        set(p[0], d.Cout, taps * (minor ? any_padded(d.Cin, ES) : d.Cin), npix);
        // Runs of k are images: the gradient's rows are then read in whole pieces.  Where the images fill their last
        // slabs badly, k runs over all pixels and the gradient is gathered like the patches.
        if (!minor && P >= VEC && 4 * P >= 3 * ((P + SK - 1) / SK * SK)) {
            p[0].K = P;
            p[0].runs = d.batch;
        }
        return 1;
    }
    const int n = step == ANY_FW ? 1 : 0, chan = step == ANY_FW ? d.Cout : d.Cin, deep = step == ANY_FW ? d.Cin : d.Cout;
    AnyPhase f[RAG_CONV_MAX];
    const int count = n ? 1 : any_phases(d, f);
    for (int i = 0; i < count; ++i) {
        const int pix = n ? npix : d.batch * f[i].qh * f[i].qw, t = n ? taps : f[i].th * f[i].tw;
        set(p[i], d.in_hwc ? pix : chan, d.in_hwc ? chan : pix, t * (minor ? any_padded(deep, ES) / VEC : deep));
    }
    return count;
}

// What a call does: by channel-minor copies of channel-major tensors or on the tensors themselves, both gradients in one
// launch (64 x 64 tiles; small layers) or one after the other, and the tiles of its products.  Looked up by the layer's geometry, since weighing the choices takes the host 1-3 us.
struct AnyPlan {
    bool turn, one;     // one: both gradients in one launch
    RagPlan first, ig;  // forward or weight gradient; input gradient
    RagBackPlan back;
    double clocks;
};
template <typename T>
static const AnyPlan &any_plan(const ConvTileDesc &d, int steps) {
    struct Entry {
        int key[17];
        AnyPlan plan;
    };
    constexpr int ENTRIES = 64, KEYS = 17;
    static thread_local Entry table[ENTRIES] = {};
    const int path = state().gemm_path;  // 7 to 9: see ptl_set_gemm_path
    const int key[KEYS] = {steps + 8 * path, d.in_hwc, d.batch, d.Cin, d.Hin, d.Win, d.Cout, d.Ho, d.Wo, d.KH, d.KW, d.sh, d.sw, d.padU, d.padL, d.padD, d.padR};
    unsigned h = 0;
    for (int i = 0; i < KEYS; ++i) h = h * 31 + (unsigned)key[i];
    Entry &e = table[(h ^ h >> 7) % ENTRIES];
    if (memcmp(e.key, key, sizeof(key)) == 0) return e.plan;
    constexpr int ES = (int)sizeof(T);
    AnyPlan best = {};
    for (int way = 0; way < 4; ++way) {
        const bool turn = (way & 1) != 0, one = way > 1, minor = d.in_hwc || turn;
        if ((turn && d.in_hwc) || (one && (path == 7 || !(steps & ANY_IG)))) continue;
        if (path > 7 && (steps & ANY_IG) && (!one || (!d.in_hwc && turn != (path == 9)))) continue;
        AnyPlan a = {};
        a.turn = turn;
        a.one = one;
        RagProd p[RAG_CONV_MAX] = {}, w[RAG_CONV_MAX] = {};
        if (one) {
            if (steps & ANY_WG) any_sizes<T>(d, ANY_WG, minor, w);
            const int n = any_sizes<T>(d, ANY_IG, minor, p);
            a.back = ragged_back_plan<T>(steps & ANY_WG ? w : nullptr, p, n, turn ? RAG_BACK_COPIES : minor ? RAG_BACK_MINOR : RAG_BACK_MAJOR);
            a.clocks = a.back.clocks;
        }
        if (!one && (steps & (ANY_FW | ANY_WG))) {
            const int n = any_sizes<T>(d, steps & (ANY_FW | ANY_WG), minor, p);
            a.first = steps & ANY_FW ? ragged_conv_plan<T>(p, n, d.in_hwc ? RAG_GK : RAG_KC, d.in_hwc ? RAG_KC : turn ? RAG_GK : RAG_XK)
                                     : ragged_conv_plan<T>(p, n, RAG_RC, minor ? RAG_GR : RAG_XR);
            a.clocks += a.first.clocks;
        }
        if (!one && (steps & ANY_IG)) {
            const int n = any_sizes<T>(d, ANY_IG, minor, p);
            a.ig = ragged_conv_plan<T>(p, n, d.in_hwc ? RAG_GK : RAG_KC, d.in_hwc ? RAG_KC : turn ? RAG_GK : RAG_XK);
            a.clocks += a.ig.clocks;
        }
        // a launch for the layouts, and the bytes it moves (clocks fitted like those of the tiles)
        if (turn || (steps == ANY_IG && !one)) a.clocks += 12500;
        if (turn) {
            const double x = steps == ANY_IG ? 0 : (double)d.batch * d.Hin * d.Win * (d.Cin + any_padded(d.Cin, ES)) * ES;
            const double y = steps == ANY_FW ? 0 : (double)d.batch * d.Ho * d.Wo * (d.Cout + any_padded(d.Cout, ES)) * ES;
            a.clocks += (x + y) / (ES == 2 ? 1500 : 2000);
        }
        if (best.clocks == 0 || a.clocks < best.clocks) best = a;
    }
    memcpy(e.key, key, sizeof(key));
    e.plan = best;
    return e.plan;
}

template <typename T>
int conv_any_fw(const ConvTileDesc &d, const void *X, const void *Wt, const void *bias, void *Y) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES;
    const int taps = d.KH * d.KW, K = d.Cin * taps, P = d.Ho * d.Wo, npix = d.batch * P;
    if (!any_fits(d, ES) || (d.in_hwc ? d.Cin < VEC : K < VEC)) return -1;
    const AnyPlan &plan = any_plan<T>(d, ANY_FW);
    const bool turn = plan.turn, minor = d.in_hwc || turn;
    state().last_conv_resident = turn ? 4 : 0;
    const int Cp = any_padded(d.Cin, ES), Kp = taps * Cp;
    RagConvArgs r = {};
    if (turn) {  // filters tap by tap, whole pieces of channels; the image channel-minor
        const size_t w_bytes = ((size_t)d.Cout * Kp * ES + 255) / 256 * 256;
        char *buf = static_cast<char *>(scratch(w_bytes + (size_t)d.batch * d.Hin * d.Win * Cp * ES));
        if (!buf) return 2;
        RagRelay &l = r.relay[0];
        r.relay_src = Wt;
        r.relays = 1;
        l.dst = buf;
        l.rows = d.Cout; l.row_s = K;
        l.outer = 1;
        l.taps = taps; l.kw = d.KW;
        l.tap_x = 1; l.tap_y = d.KW;
        l.inner = Cp; l.lim = d.Cin; l.inner_s = taps;
        const RagTurn t = {X, buf + w_bytes, d.batch, d.Cin, Cp, d.Hin * d.Win};
        if (int rc = ragged_relay<T>(r, &t, 1)) return rc;
        r.relays = 0;
        Wt = buf;
        X = t.dst;
    }
    RagProd &p = r.p[0];
    r.count = any_sizes<T>(d, ANY_FW, minor, r.p);
    p.C = Y;
    p.bias = bias;
    const AnyImage img = {turn ? Cp : d.Cin, d.Hin, d.Win, minor, (long long)d.batch * d.Cin * d.Hin * d.Win * ES};
    RagOp &patch = d.in_hwc ? p.a : p.b, &weight = d.in_hwc ? p.b : p.a;
    if (any_geo<T>(r.geo[0], patch, X, img, d.Ho, d.Wo, -d.padU, -d.padL, d.sh, d.sw, d.KH, d.KW, 1)) return -1;
    patch.rows = npix;
    weight = any_rows<T>(Wt, d.Cout, (long long)(minor ? Kp : K) * ES);
    if (d.in_hwc) {
        p.cn = rag_axis(npix, d.Cout);
        p.cm = rag_axis(d.Cout, 1);
        if (Kp != K) {  // channels that are no whole pieces: filters in place, their rows as the pixels of images of KH x KW
            const AnyImage filter = {d.Cin, d.KH, d.KW, 1, (long long)d.Cout * K * ES};
            if (any_geo<T>(r.geo_a, weight, Wt, filter, 1 << 30, 1 << 30, 0, 0, 0, 0, d.KH, d.KW, 1)) return -1;
            r.geo_a.px = (unsigned)(K * ES);
            return ragged_conv<T>(r, RAG_GK, RAG_GK, plan.first);
        }
        return ragged_conv<T>(r, RAG_GK, RAG_KC, plan.first);
    }
    p.bias_n = 1;
    p.cn = rag_axis(d.Cout, P);
    p.cm = rag_axis2(P, 1, d.Cout * P);
    return ragged_conv<T>(r, RAG_KC, turn ? RAG_GK : RAG_XK, plan.first);
}

// The filters of a phase in place, for the input gradient: as a patch matrix whose pixels are the input channels and whose
// channels the output channels (channel-major), or by tap and output channel (channel-minor).
template <typename T>
static void any_filters(const ConvTileDesc &d, const void *Wt, const AnyPhase &f, RagGeo &g, RagOp &o) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES;
    const int taps = d.KH * d.KW, t = f.th * f.tw, c = d.in_hwc ? d.Cin : 1;
    const int tap_at = (f.ky * d.KW + f.kx) * c * ES, tap_y = d.sh * d.KW * c * ES, tap_x = d.sw * c * ES;
    o = {};
    o.p = static_cast<const char *>(Wt) + tap_at;
    o.rows = d.Cin;
    g.plane = (unsigned)(d.Cin * taps * ES);
    g.d_kw = rag_div(f.tw);
    if (d.in_hwc) {
        g.d_cb = rag_div((d.Cout + VEC - 1) / VEC);
        g.py = (unsigned)tap_y;
        g.px = (unsigned)tap_x;
        g.size = (unsigned)d.Cout;
        return;
    }
    g.d_x = g.d_y = rag_div(1 << 30);
    g.px = (unsigned)(taps * ES);
    g.ty = g.tx = 1;
    g.H = g.W = 1 << 30;
    g.d_t = rag_div(t);
    for (int i = 0; i < t; i += f.tw) g.every_row |= 1u << i;
    for (int i = 0; i < 32 && t > 0; i += t) g.every_channel |= 1u << i;
    g.all_taps = (1u << t) - 1u;
    g.size = (unsigned)((long long)d.Cout * d.Cin * taps * ES - tap_at);
    for (int j = 0; j < RAG_TAB && t > 0; ++j) g.tab[j] = j / t * (int)g.plane + j % t / f.tw * tap_y + j % t % f.tw * tap_x;
}

// The products of the input gradient, one per phase, and the filters they read: in place (geometry to `in_place`) or re-laid at
// W as `filters` says.  turn: dY is the channel-minor copy of a channel-major gradient.
template <typename T>
static int any_input_gradient(const ConvTileDesc &d, const void *dY, const void *Wt, void *dX, bool turn, char *W, RagConvArgs &r, RagConvArgs &filters,
                              RagGeo *in_place) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES;
    const bool minor = d.in_hwc || turn;
    const int taps = d.KH * d.KW, Cp = any_padded(d.Cout, ES), inner = minor ? Cp : 1, outer = minor ? 1 : d.Cout;
    const AnyImage img = {turn ? Cp : d.Cout, d.Ho, d.Wo, minor, (long long)d.batch * d.Cout * d.Ho * d.Wo * ES};
    filters.relay_src = Wt;
    AnyPhase phase[RAG_CONV_MAX];
    any_phases(d, phase);
    r.count = any_sizes<T>(d, ANY_IG, minor, r.p);
    for (int i = 0; i < r.count; ++i) {
        const AnyPhase &f = phase[i];
        const int t = f.th * f.tw, K = t * outer * inner;
        if (t > 0 && K < VEC) return -1;
        RagProd &p = r.p[i];
        RagOp &patch = d.in_hwc ? p.a : p.b, &weight = d.in_hwc ? p.b : p.a;
        if (any_geo<T>(r.geo[i], patch, dY, img, f.qh, f.qw, f.y0, f.x0, 1, 1, f.th, f.tw, -1)) return -1;
        patch.rows = d.batch * f.qh * f.qw;
        if (in_place) any_filters<T>(d, Wt, f, in_place[i], weight);
        else weight = any_rows<T>(W, d.Cin, (long long)K * ES);
        const int pix = d.in_hwc ? d.Cin : 1, img_n = d.Cin * d.Hin * d.Win;
        p.C = static_cast<T *>(dX) + (f.ph * d.Win + f.pw) * pix;
        const RagAxis pixels = d.sh == 1 && d.sw == 1 ? rag_axis2(d.Hin * d.Win, pix, img_n) : rag_axis3(f.qw, f.qh, d.sw * pix, d.sh * d.Win * pix, img_n);
        const RagAxis chans = rag_axis(d.Cin, d.in_hwc ? 1 : d.Hin * d.Win);
        p.cn = d.in_hwc ? pixels : chans;
        p.cm = d.in_hwc ? chans : pixels;
        if (t == 0 || in_place) continue;
        RagRelay &l = filters.relay[filters.relays++];
        const int c = d.in_hwc ? d.Cin : 1;  // from tap to tap
        l.dst = W;
        l.rows = d.Cin; l.row_s = d.in_hwc ? 1 : taps;
        l.outer = outer; l.outer_s = d.Cin * taps;
        l.taps = t; l.kw = f.tw; l.tap_at = (f.ky * d.KW + f.kx) * c; l.tap_y = d.sh * d.KW * c; l.tap_x = d.sw * c;
        l.inner = inner; l.lim = minor ? d.Cout : 1; l.inner_s = d.Cin * taps;
        W += (size_t)d.Cin * K * ES;
    }
    return 0;
}

template <typename T>
int conv_any_bw(const ConvTileDesc &d, const void *X, const void *dY, const void *Wt, void *dW, void *dX, void *db) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES, SK = 128 / ES;
    const int taps = d.KH * d.KW, P = d.Ho * d.Wo, npix = d.batch * P;
    if (!any_fits(d, ES) || (d.in_hwc && (d.Cin < VEC || d.Cout < VEC))) return -1;
    const AnyPlan &plan = any_plan<T>(d, (dW ? ANY_WG : 0) | (dX ? ANY_IG : 0));
    const bool turn = plan.turn && d.Cout >= VEC, minor = d.in_hwc || turn;
    state().last_conv_resident = turn ? 4 : 0;
    const int Cip = any_padded(d.Cin, ES), Cop = any_padded(d.Cout, ES);
    // scratch: the filters as the input gradient reads them; channel-minor copies of the gradient and of the input
    const bool relaid = dX && (turn || !plan.one);
    const size_t w_bytes = relaid ? ((size_t)d.Cin * taps * (minor ? Cop : d.Cout) * ES + 255) / 256 * 256 : 0;
    const size_t y_bytes = turn ? ((size_t)npix * Cop * ES + 255) / 256 * 256 : 0, x_bytes = turn && dW ? (size_t)d.batch * d.Hin * d.Win * Cip * ES : 0;
    char *buf = nullptr;
    if (w_bytes + y_bytes + x_bytes && !(buf = static_cast<char *>(scratch(w_bytes + y_bytes + x_bytes)))) return 2;
    RagTurn t[2];
    if (turn) {
        t[0] = {dY, buf + w_bytes, d.batch, d.Cout, Cop, P};
        t[1] = {X, buf + w_bytes + y_bytes, d.batch, d.Cin, Cip, d.Hin * d.Win};
        dY = t[0].dst;
        X = t[1].dst;
    }
    RagConvArgs w = {}, x = {};
    RagProd &p = w.p[0];
    int am = RAG_RC, bm = RAG_GR;
    if (dW) {
        w.count = any_sizes<T>(d, ANY_WG, minor, w.p);
        p.C = dW;
        p.row_sum = db;
        p.cn = rag_axis(d.Cout, d.Cin * taps);
        const AnyImage img = {turn ? Cip : d.Cin, d.Hin, d.Win, minor, (long long)d.batch * d.Cin * d.Hin * d.Win * ES};
        if (any_geo<T>(w.geo[0], p.b, X, img, d.Ho, d.Wo, -d.padU, -d.padL, d.sh, d.sw, d.KH, d.KW, 1)) return -1;
        if (minor) {
            p.a.p = static_cast<const char *>(dY);
            p.a.rows = d.Cout;
            p.a.k_b = (unsigned)((turn ? Cop : d.Cout) * ES);
            p.b.rows = p.M;
            p.cm = d.in_hwc ? rag_axis2(Cip, 1, d.Cin) : rag_axis2(Cip, taps, 1);
            p.cm.lim = d.Cin;
        } else {
            p.b.rows = p.M;
            p.cm = rag_axis(p.M, 1);
            bm = RAG_XR;
            if (P >= VEC && p.runs == d.batch) {
                am = RAG_KC;
                p.a = any_rows<T>(dY, d.Cout, (long long)P * ES);
                p.a.run_b = (long long)d.Cout * P * ES;
            } else {
                am = RAG_XR;
                const AnyImage flat = {1, 1 << 30, P, 0, (long long)d.batch * d.Cout * P * ES};  // (its rows are the samples)
                if (any_geo<T>(w.geo_a, p.a, dY, flat, 1 << 30, P, 0, 0, 1, 1, 1, 1, 1)) return -1;
                w.geo_a.py = (unsigned)(d.Cout * P * ES);
                w.geo_a.plane = (unsigned)(P * ES);
                for (int j = 0; j < RAG_TAB; ++j) w.geo_a.tab[j] = j * P * ES;
                p.a.rows = d.Cout;
            }
        }
    }
    RagGeo in_place[RAG_CONV_MAX] = {};
    if (dX)
        if (int rc = any_input_gradient<T>(d, dY, Wt, dX, turn, buf, x, w, relaid ? nullptr : in_place)) return rc;
    // the filters: together with the channel-minor copies, else by spare blocks of the weight gradient's launch
    if (turn || (!dW && relaid)) {
        if (int rc = ragged_relay<T>(w, t, turn ? (dW ? 2 : 1) : 0)) return rc;
        w.relays = 0;
    }
    if (plan.one && dX) return ragged_back<T>(w, x, in_place, turn ? RAG_BACK_COPIES : minor ? RAG_BACK_MINOR : RAG_BACK_MAJOR, am, plan.back);
    if (dW)
        if (int rc = ragged_conv<T>(w, am, bm, plan.first)) return rc;
    return dX ? ragged_conv<T>(x, d.in_hwc ? RAG_GK : RAG_KC, d.in_hwc ? RAG_KC : turn ? RAG_GK : RAG_XK, plan.ig) : 0;
}

// 1 x 1 layers of unit stride without padding: products of matrices.  -1: rows or images shorter than a piece.
template <typename T>
int conv_point_fw(const ConvTileDesc &d, const void *X, const void *Wt, const void *bias, void *Y) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES;
    const int P = d.Hin * d.Win;
    if (!any_fits(d, ES) || P < VEC || d.Cin < VEC) return -1;
    RagArgs r = {};
    RagProd &p = r.p[0];
    r.count = p.runs = p.outer = 1;
    p.K = d.Cin;
    p.C = Y;
    p.bias = bias;
    RagOp &pixels = d.in_hwc ? p.a : p.b, &weight = d.in_hwc ? p.b : p.a;
    weight = any_rows<T>(Wt, d.Cout, (long long)d.Cin * ES);
    if (d.in_hwc) {
        p.N = d.batch * P;
        p.M = p.m_in = d.Cout;
        pixels = any_rows<T>(X, p.N, (long long)d.Cin * ES);
        p.cn = rag_axis(p.N, d.Cout);
        p.cm = rag_axis(d.Cout, 1);
        return ragged<T>(r, RAG_KC, RAG_KC, RAG_KC, RAG_KC);
    }
    p.N = d.Cout;
    p.M = d.batch * P;
    p.m_in = P;
    p.outer = d.batch;
    pixels = any_rows<T>(X, P, 0);
    pixels.k_b = (unsigned)(P * ES);
    pixels.outer_b = (long long)d.Cin * P * ES;
    p.cn = rag_axis(d.Cout, P);
    p.cm = rag_axis2(P, 1, d.Cout * P);
    p.bias_n = 1;
    return ragged<T>(r, RAG_KC, RAG_RC, RAG_KC, RAG_RC);
}
template int conv_point_fw<float>(const ConvTileDesc &, const void *, const void *, const void *, void *);
template int conv_point_fw<half_t>(const ConvTileDesc &, const void *, const void *, const void *, void *);

// Both gradients in one launch, channel-major tensors.
template <typename T>
int conv_point_bw(const ConvTileDesc &d, const void *X, const void *dY, const void *Wt, void *dW, void *dX, void *db) {
    constexpr int ES = (int)sizeof(T), VEC = 16 / ES;
    const int P = d.Hin * d.Win;
    if (!any_fits(d, ES) || P < VEC || d.Cin < VEC) return -1;
    RagConvArgs w = {}, x = {};
    RagProd &p = w.p[0], &q = x.p[0];
    w.count = x.count = 1;
    p.N = d.Cout;
    p.M = p.m_in = d.Cin;
    p.K = P;
    p.runs = d.batch;
    p.a = any_rows<T>(dY, d.Cout, (long long)P * ES);
    p.a.run_b = (long long)d.Cout * P * ES;
    p.b = any_rows<T>(X, d.Cin, (long long)P * ES);
    p.b.run_b = (long long)d.Cin * P * ES;
    p.C = dW;
    p.row_sum = db;
    p.cn = rag_axis(d.Cout, d.Cin);
    p.cm = rag_axis(d.Cin, 1);
    q.N = d.Cin;
    q.M = d.batch * P;
    q.m_in = P;
    q.K = d.Cout;
    q.a = any_rows<T>(Wt, d.Cin, 0);
    q.a.k_b = (unsigned)(d.Cin * ES);
    q.b = any_rows<T>(dY, P, 0);
    q.b.k_b = (unsigned)(P * ES);
    q.b.outer_b = (long long)d.Cout * P * ES;
    q.C = dX;
    q.cn = rag_axis(d.Cin, P);
    q.cm = rag_axis2(P, 1, d.Cin * P);
    p.outer = q.runs = 1;
    q.outer = d.batch;
    const RagBackPlan plan = ragged_back_plan<T>(&p, &q, 1, RAG_BACK_POINT);
    state().last_conv_resident = 0;
    const RagGeo none = {};
    return ragged_back<T>(w, x, &none, RAG_BACK_POINT, RAG_KC, plan);
}

template int conv_point_bw<float>(const ConvTileDesc &, const void *, const void *, const void *, void *, void *, void *);
template int conv_point_bw<half_t>(const ConvTileDesc &, const void *, const void *, const void *, void *, void *, void *);
template int conv_any_fw<float>(const ConvTileDesc &, const void *, const void *, const void *, void *);
template int conv_any_fw<half_t>(const ConvTileDesc &, const void *, const void *, const void *, void *);
template int conv_any_bw<float>(const ConvTileDesc &, const void *, const void *, const void *, void *, void *, void *);
template int conv_any_bw<half_t>(const ConvTileDesc &, const void *, const void *, const void *, void *, void *, void *);

}  // namespace ptl
