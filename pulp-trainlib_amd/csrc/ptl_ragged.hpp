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

// How the 16-byte chunks of an operand are found.  KC and RC: a matrix whose rows (KC) or whose k columns (RC) are
// contiguous.  GK and GR: an implicit patch matrix over a channel-minor or channel-blocked tensor, whose chunks are VEC
// channels of one tap at one pixel - with pixels as the rows (GK) or as the contraction index (GR).
enum RagMode : int { RAG_KC = 0, RAG_RC = 1, RAG_GK = 2, RAG_GR = 3 };

struct RagOp {
    const char *p;     // first element
    int rows;          // extent along the output
    unsigned row_b;    // KC: bytes from row to row
    unsigned k_b;      // RC: bytes from k to k
    long long run_b;   // bytes from one run of k to the next
    long long outer_b; // RC: bytes between the outer digits of the rows
    // GK, GR: pixel = (b, y, x) -> bytes, chunk = (tap row, tap column, channel chunk) -> bytes
    RagDiv d_x, d_y;         // extents of x and y
    unsigned px, py, pb;
    RagDiv d_cb, d_kw;       // channel chunks per tap, taps per row
    unsigned tc, tx, ty;
    int chunks;              // taps x channel chunks
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
    int N, M, K;       // K: k per run (GR: pixels, GK: 128-byte slabs of chunks are counted from b.chunks)
    int runs;          // runs of K (KC / RC operands)
    int outer, m_in;   // RC second operand: M = outer x m_in, tiles stay inside one outer digit (outer == 1: m_in == M)
    const void *bias;  // added per n (bias_n) or per m
    int bias_n;
    void *row_sum;     // sum over k of a(n, k), as an extra column of ones in b (RC / GR second operand)
    // set by the launcher
    float *ws;         // partial sums [split][N][pitch]
    int pitch, splits, slabs_per_split;
    int tiles_n, tiles_m, tiles_in;  // tiles along n, along m, along m inside one outer digit
};

constexpr int RAG_MAX = 5;
struct RagArgs {
    RagProd p[RAG_MAX];
    int first[RAG_MAX + 1];  // first workgroup of each product
    int count;
};

// The products in one launch (plus one for their partial sums where the contraction is split).  The first product has
// the modes (a0, b0), the others (a1, b1).  0 = launched, -1 = no such combination of modes, 2 = a HIP failure.
template <typename T>
int ragged(RagArgs &r, int a0, int b0, int a1, int b1);

}  // namespace ptl
