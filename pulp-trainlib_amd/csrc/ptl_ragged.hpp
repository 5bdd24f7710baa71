// MFMA product for tensors of any size and alignment: host-side description (kernel: ptl_ragged.inc).
#pragma once
#include "ptl_common.hpp"

namespace ptl {

// n / d for n < 2^31 by a multiplication and a shift (d == 1: m == 0 stands for the identity).
struct RagDiv {
    unsigned d, m;
    int s;
};
inline RagDiv rag_div(long long dv) {
    RagDiv r = {(unsigned)(dv < 1 ? 1 : dv), 0u, 0};
    if (r.d == 1) return r;
    int l = 1;
    while (((unsigned long long)1 << l) < r.d) ++l;
    r.m = (unsigned)((((unsigned long long)1 << (31 + l)) + r.d - 1) / r.d);
    r.s = l - 1;
    return r;
}
__device__ inline unsigned rag_quot(unsigned n, const RagDiv &d) { return d.m ? __umulhi(n, d.m) >> d.s : n; }

// How an operand's tile is filled.  KC and RC: 16-byte pieces of a matrix whose rows (KC) or whose k columns (RC) are
// contiguous.  The others are implicit patch matrices (RagGeo): XK and XR gather a channel-major tensor element by element,
// neighbouring lanes at neighbouring pixels, with pixels as the rows and (channel, tap) as k (XK) or the other way round
// (XR); GK and GR read channel-minor tensors in pieces of VEC channels of one tap at one pixel, with pixels as the rows
// and (tap, piece) as k (GK) or the other way round (GR).  WR: the filters of a channel-minor layer in place, input channels
// (contiguous) as the rows and (tap, piece of output channels) as k, beside GK.
enum RagMode : int { RAG_KC = 0, RAG_RC = 1, RAG_GK = 2, RAG_GR = 3, RAG_XK = 4, RAG_XR = 5, RAG_WR = 6 };

struct RagOp {
    const char *p;     // first element (XK, XR: see RagGeo)
    int rows;          // extent along the output (GR: taps x pieces x VEC)
    unsigned row_b;    // KC: bytes from row to row; RC with `pad`: rows in all
    unsigned k_b;      // RC: bytes from k to k
    RagDiv pad;        // RC, d > 0: the outer digits follow each other, each filled up to so many rows (rag_row_up)
    long long run_b;   // bytes from one run of k to the next (KC, RC)
    long long outer_b; // RC: bytes between the outer digits of the rows
};

// An implicit patch matrix: pixel q = (b, qy, qx), tap t = (jy, jx), element at row qy*sy + y0 + ty*jy and column
// qx*sx + x0 + tx*jx of channel c of image b, zero outside of the H x W image.  ty = tx = 1 for a forward pass, -1 for the
// input gradient.  Offsets are unsigned: the tensor pointer is moved back by what the smallest of them would lack.
// XK also reads filters in place, the input channels as its pixels and the output channels as its channels; WR has the
// bytes from tap to tap in py and px, from output channel to output channel in plane, and in size how many there are.
constexpr int RAG_TAPS = 25;          // one validity bit per tap and for the seven taps after the last of a channel
constexpr int RAG_TAB = RAG_TAPS + 7;
struct RagGeo {
    RagDiv d_x, d_y;        // extents of qx and qy
    unsigned pb, py, px;    // bytes per step of b, qy, qx
    int y0, x0, sy, sx, ty, tx, H, W;
    RagDiv d_t, d_kw;       // taps, taps per row
    RagDiv d_cb;            // GK, GR: pieces per tap
    unsigned every_row, every_channel, all_taps;  // bit 0 of every row of taps, of every channel's taps (GK: bit 0); the taps
    unsigned plane;         // XK, XR: bytes from channel to channel
    unsigned size;          // XK, XR: bytes from the moved pointer to the end of the tensor
    unsigned cut;           // GK, GR: bytes that the last piece of a tap lacks
    const char *zeros;      // GK, GR: 16 zero bytes
    int tab[RAG_TAB];       // bytes of tap t; XK, XR: of entry j = tap j % taps of channel j / taps
};

// Output axis: index -> (q2, q1, q0) with the radices of d1 and d0 -> elements.  q0 below `lim` only.
struct RagAxis {
    RagDiv d0, d1;
    int s0, s1, s2, lim;
};
inline RagAxis rag_axis(int n, int stride) { return {rag_div(n > 0 ? n : 1), rag_div(1), stride, 0, 0, n}; }
inline RagAxis rag_axis2(int d0, int s0, int s1) { return {rag_div(d0), rag_div(1 << 30), s0, s1, 0, d0}; }
inline RagAxis rag_axis3(int d0, int d1, int s0, int s1, int s2) { return {rag_div(d0), rag_div(d1), s0, s1, s2, d0}; }

struct RagProd {
    RagOp a, b;        // C(n, m) = sum over runs and k of a(n, k) * b(m, k)
    void *C;
    RagAxis cn, cm;
    int N, M, K;       // K: k per run (GK: pieces)
    int runs;          // runs of K (with a patch matrix: run r is image r)
    int outer, m_in;   // RC second operand: M = outer x m_in, tiles stay inside one outer digit (outer == 1: m_in == M)
    const void *bias;  // added per n (bias_n) or per m
    int bias_n;
    int whole_k;       // the contraction is not split
    int add;           // C keeps what it holds, the product is added to it
    void *row_sum;     // sum over k of a(n, k); in the first product of (RC, RC) before (KC, RC), and with b gathered along k
    // set by the launcher
    float *ws;         // partial sums [split][N][pitch], behind them those of the row sums [split][N]
    int pitch, splits, slabs_per_split;
    int tiles_n, tiles_m, tiles_in;  // tiles along n, along m, along m inside one outer digit
};

constexpr int RAG_MAX = 5;
struct RagArgs {
    int first[RAG_MAX + 1];  // first workgroup of each product
    int count;
    int shape;  // 32, 64: that tile, whatever it costs (sums in the same order at every size); 0: the cheapest
    // of the first product of (KC, RC) before (KC, KC) only: up to three runs of k lie anywhere, run r + 1 hop_a[r],
    // hop_b[r] bytes behind run r (its run_b is not used)
    long long hop_a[2], hop_b[2];
    RagProd p[RAG_MAX];
};

struct RagSums {  // the products whose contraction was split
    int first[6];
    int count;
    int sums;  // the one whose row sums are wanted, or -1
    RagProd p[5];
};

// The products in one launch (plus one for their partial sums where the contraction is split).  The first product has
// the modes (a0, b0), the others (a1, b1).  0 = launched, -1 = no such combination of modes, 2 = a HIP failure.
template <typename T>
int ragged(RagArgs &r, int a0, int b0, int a1, int b1);

// Filters re-laid for a product: dst[row][k], k = (outer, tap, inner), from src at row*row_s + outer*outer_s + inner*inner_s
// + tap_at + jy*tap_y + jx*tap_x; inner values from `lim` on are zeros.  All in elements.
struct RagRelay {
    void *dst;
    int rows, outer, taps, inner, lim, kw;
    int row_s, outer_s, inner_s, tap_at, tap_y, tap_x;
    RagDiv by_k, by_inner, by_taps, by_kw;  // set by the launcher
};

// A channel-major tensor re-laid channel-minor: dst[b][pixel][cp] from src[b][channel][pixel], zeros from channel c on; cp is
// a whole number of 16-byte pieces.
struct RagTurn {
    const void *src;
    void *dst;
    int batch, c, cp, pix;
};

// Products with patch matrices: N of them, one or the phases of a strided input gradient (up to four).
constexpr int RAG_CONV_MAX = 4;
template <int N>
struct RagConvOf {
    int first[N + 1];
    int count;
    int relays, relay_first[RAG_CONV_MAX + 1];
    RagProd p[N];
    RagGeo geo[N];          // of each product's patch matrix
    RagGeo geo_a;           // of the other operand where it is gathered too (one product): a gradient (XR), filters (GK, GK)
    const void *relay_src;  // blocks behind the last product re-lay filters for a later product
    RagRelay relay[RAG_CONV_MAX];
};
typedef RagConvOf<RAG_CONV_MAX> RagConvArgs;
// The tiles and slabs per workgroup that ragged_conv() would choose for the products (of which sizes and runs count), and the clocks of
// 2.4 GHz that this would take.
struct RagPlan {
    int shape, per_wg;
    double clocks;
};
template <typename T>
RagPlan ragged_conv_plan(const RagProd *p, int count, int a, int b);
template <typename T>
int ragged_conv(RagConvArgs &r, int a, int b, const RagPlan &plan);
// Both gradients of a layer in one launch (plus one for partial sums): the weight gradient of w (modes a, b; none where its
// count is 0), then the products of x, whose filters are read in place as f says - channel-major by XK, channel-minor by WR -
// or, where the tensors of x are channel-minor copies (KC, GK), re-laid.  POINT: 1 x 1 layers of unit stride on channel-major
// tensors, which are matrices (KC, KC before RC, RC).
struct RagBackPlan {
    int per_w, per_x;  // slabs per workgroup
    double clocks;
};
enum RagBack : int { RAG_BACK_MAJOR = 0, RAG_BACK_MINOR = 1, RAG_BACK_COPIES = 2, RAG_BACK_POINT = 3 };
template <typename T>
RagBackPlan ragged_back_plan(const RagProd *w, const RagProd *x, int count, RagBack kind);
template <typename T>
int ragged_back(RagConvArgs &w, RagConvArgs &x, const RagGeo *f, RagBack kind, int a, const RagBackPlan &plan);
// The re-laying alone, filters of r and tensors (n <= 2).
template <typename T>
int ragged_relay(RagConvArgs &r, const RagTurn *turn, int n);

// C[N][M] = A[N][K] * B[M][K]^T (+ bias[M]) with the contraction shared out over the waves of a tile; K >= 16 bytes.
template <typename T>
int ragged_deep(const T *A, const T *B, T *C, int N, int M, int K, const T *bias);

}  // namespace ptl
