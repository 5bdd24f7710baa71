// Multi-head self-attention training step, fp32 (lib/sources/pulp_mhsa_fp32.c:20 forward, :648 backward)
// and the row softmax it is built on (lib/sources/pulp_act_fp32.c:187, :335).
//
// Tensors (L = sequence length, E = token size, F = heads x head size H; tokens are COLUMNS):
//   input/output E x L, q/k/v/attention_map F x L, softmax_buffer heads x L x L (row = query, column = key),
//   coeff_in_* stored E x F with gradients F x E, coeff_out E x F.
// The reference writes a transposed copy of an operand into a scratch buffer before most products; here the
// projections run on the index-map GEMM (which reads operands in place in either orientation) and the
// per-head part runs in three fused kernels that keep a 32-query (or 32-key) tile of the L x L score matrix
// in LDS:
//   forward      scores -> approximate-exponential softmax -> probabilities (saved) -> value mix
//   backward I   per query tile: dP = dA^T v, softmax backward, dq
//   backward II  per key tile:   dv = dA P, dk = q dS
// MFMA: v_mfma_f32_32x32x2_f32.  Rows of the F x L tensors are L floats long (197 in ViT-Tiny), so nothing
// here assumes 16-byte alignment of a row: global accesses are 4-byte, consecutive lanes on consecutive
// addresses.
#include <float.h>

#include <type_traits>

#include "ptl_api.h"
#include "ptl_gemm_async.hpp"
#include "ptl_gemm_async.inc"
#include "ptl_host.hpp"
#include "ptl_internal.h"
#include "ptl_ragged.hpp"
#include "ptl_structs.h"

namespace ptl {

typedef float mh_f32x16 __attribute__((ext_vector_type(16)));

constexpr int ATT_NT = 256;  // threads of an attention workgroup (4 waves)
constexpr int ATT_CK = 64;   // contraction columns staged per chunk
constexpr int ATT_VP = ATT_CK + 1;
constexpr int ATT_RP = 33;   // pitch of a parked 32 x 32 accumulator tile

// exp(x) by writing a scaled, shifted x into the exponent field (fastexp_gist,
// lib/sources/pulp_train_utils_fp32.c:1223, constants lib/include/pulp_train_defines.h:85-88).
// Multiply and add are rounded separately, as in the reference's golden model.
__device__ inline float fastexp_gist(float x) {
    x = __fadd_rn(__fmul_rn(12102203.17133801f, x), 1064986823.010288f);
    if (x < 8388608.f || x > 2139095040.f) x = (x < 8388608.f) ? 0.0f : 2139095040.f;
    return __builtin_bit_cast(float, (uint32_t)x);
}

// The same for x <= 0 or NaN, which have no upper end to be kept from.
__device__ inline float fastexp_below(float x) {
    x = __fadd_rn(__fmul_rn(12102203.17133801f, x), 1064986823.010288f);
    return x < 8388608.f ? 0.f : __builtin_bit_cast(float, (uint32_t)x);
}

// 1/sqrt by the magic-constant estimate and one Newton step (q_rsqrt,
// lib/sources/pulp_train_utils_fp32.c:1234; 32-bit integer as on the reference's target).
static float q_rsqrt_host(float number) {
    float x2 = number * 0.5f, y = number;
    int32_t i = __builtin_bit_cast(int32_t, y);
    i = 0x5f3759df - (i >> 1);
    y = __builtin_bit_cast(float, i);
    return y * (1.5f - (x2 * y * y));
}

// Reductions over the wave in registers (shifts inside rows of 16 lanes, then from row to row; the last lane has the
// result): a chain of six shuffles through LDS took most of the softmax phase.
template <int CTRL>
__device__ inline float dpp_from(float v, float otherwise) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, otherwise), __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
__device__ inline float last_lane(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63)); }
__device__ inline float wave_max(float v) {
    v = fmaxf(v, dpp_from<0x111>(v, -FLT_MAX));  // row_shr 1, 2, 4, 8
    v = fmaxf(v, dpp_from<0x112>(v, -FLT_MAX));
    v = fmaxf(v, dpp_from<0x114>(v, -FLT_MAX));
    v = fmaxf(v, dpp_from<0x118>(v, -FLT_MAX));
    v = fmaxf(v, dpp_from<0x142>(v, -FLT_MAX));  // row_bcast 15, 31
    v = fmaxf(v, dpp_from<0x143>(v, -FLT_MAX));
    return last_lane(v);
}
__device__ inline float wave_sum(float v) {
    v += dpp_from<0x111>(v, 0.f);
    v += dpp_from<0x112>(v, 0.f);
    v += dpp_from<0x114>(v, 0.f);
    v += dpp_from<0x118>(v, 0.f);
    // (a broadcast reaches rows that have their part already: rows 1 and 3, then 2 and 3, take it)
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false));
    return last_lane(v);
}

// S[r][c] = scale * sum_d R[d][r0 + r] * Cm[d][c] for 32 rows r and every column c < L, into the LDS tile
// S[32][LP].  R and Cm are [H][L] in global memory (consecutive lanes read consecutive r or c).  Each wave owns
// every fourth 32-column block; the 32 row fragments stay in registers for all of them.
template <int HMAX>
__device__ inline void scores_to_lds(const float *__restrict__ R, const float *__restrict__ Cm, int L, int H,
                                     int r0, float scale, float *S, int LP) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    constexpr int STEPS = HMAX / 2;
    float af[STEPS];
    const int r = r0 + l32;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int d = 2 * s + half;
        af[s] = (r < L && d < H) ? R[(size_t)d * L + r] : 0.f;
    }
    const int CB = (L + 31) / 32;
    for (int cb = wave; cb < CB; cb += 4) {
        const int c = cb * 32 + l32;
        float bf[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int d = 2 * s + half;
            bf[s] = (c < L && d < H) ? Cm[(size_t)d * L + c] : 0.f;
        }
        mh_f32x16 acc = {0};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[s], bf[s], acc, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) S[(8 * (v / 4) + 4 * half + (v % 4)) * LP + c] = acc[v] * scale;
    }
}

// out[d][r0 + r] = sum_c V[d][c] * S[r][c] for d < H, with S the LDS tile (columns >= L hold zeros up to the
// chunk boundary) and V [H][L] in global memory, staged through LDS in chunks of ATT_CK columns (fetched
// row-wise, read column-wise).  The 32-row blocks of d and, when there are fewer than four of them, ranges
// of the contraction are dealt to the four waves; partial tiles meet in LDS.
template <int HMAX>
__device__ inline void mix_from_lds(const float *__restrict__ V, const float *S, int LP, int L, int H, int r0,
                                    float *__restrict__ out, float *vbuf, float *red) {
    constexpr int DB = HMAX / 32, KS = 4 / DB;
    constexpr int PER = HMAX * ATT_CK / ATT_NT;
    constexpr int SPW = (ATT_CK / 2) / KS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int db = wave % DB, ks = wave / DB;
    float stage[PER];
    auto fetch = [&](int c0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + ATT_NT * i, d = idx >> 6, c = c0 + (idx & 63);
            stage[i] = (d < H && c < L) ? V[(size_t)d * L + c] : 0.f;
        }
    };
    const int chunks = (L + ATT_CK - 1) / ATT_CK;
    mh_f32x16 acc = {0};
    fetch(0);
    for (int ch = 0; ch < chunks; ++ch) {
        __syncthreads();  // the previous chunk has been consumed
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + ATT_NT * i;
            vbuf[(idx >> 6) * ATT_VP + (idx & 63)] = stage[i];
        }
        __syncthreads();
        if (ch + 1 < chunks) fetch((ch + 1) * ATT_CK);
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const int kk = 2 * (ks * SPW + s) + half;
            const float a = vbuf[(db * 32 + l32) * ATT_VP + kk];
            const float b = S[l32 * LP + ch * ATT_CK + kk];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) red[(wave * 32 + 8 * (v / 4) + 4 * half + (v % 4)) * ATT_RP + l32] = acc[v];
    __syncthreads();
    for (int idx = tid; idx < HMAX * 32; idx += ATT_NT) {
        const int d = idx >> 5, rr = idx & 31;
        float s = 0.f;
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2) s += red[((k2 * DB + (d >> 5)) * 32 + (d & 31)) * ATT_RP + rr];
        if (d < H && r0 + rr < L) out[(size_t)d * L + r0 + rr] = s;
    }
}

// ---------------------------------------------------------------------------------------------------------
// Tile loader: element (i, j), i < nrows, j < ncols (a multiple of 4), comes from g[i*gstride + j] when
// i < rvalid and j < cvalid and is zero otherwise; it lands at lds[i*pitch + j].  Each lane moves four
// consecutive columns with one 16-byte LDS-DMA load (global addresses need only 4-byte alignment, so rows of
// odd length are fine); a vector that straddles the end of a row is left to tile_edge_load/store, so
// nothing is ever read outside [0, rvalid) x [0, cvalid).  Two shapes: 32-column tiles stored with pitch 32
// (eight rows per instruction) and long rows (up to 256 columns per instruction, any pitch that is a multiple
// of 4).  Work is dealt to the NW waves of the workgroup; completion = the caller's vmcnt wait + barrier.
template <int NW>
__device__ inline void tile_dma(const float *__restrict__ g, long long gstride, int nrows, int ncols, int rvalid,
                                int cvalid, float *lds, int pitch, const float *zero, int wave, int lane) {
    const unsigned lds_addr = (unsigned)(uintptr_t)(lds_char *)lds;
    int ninstr, rows_per, lanes_per_row, segs;
    if (ncols == 32 && pitch == 32) {
        rows_per = 8;
        lanes_per_row = 8;
        segs = 1;
        ninstr = (nrows + 7) >> 3;
    } else {
        rows_per = 1;
        lanes_per_row = 64;
        segs = (ncols + 255) >> 8;
        ninstr = nrows * segs;
    }
    for (int j = wave; j < ninstr; j += NW) {
        int i, col;
        unsigned m0;
        if (rows_per == 8) {
            i = j * 8 + (lane >> 3);
            col = (lane & 7) * 4;
            m0 = lds_addr + (unsigned)j * 1024u;
        } else {
            const int seg = j % segs;
            i = j / segs;
            col = seg * 256 + lane * 4;
            m0 = lds_addr + ((unsigned)i * pitch + seg * 256) * 4u;
        }
        if (i >= nrows || col >= ncols) continue;
        const bool row_ok = i < rvalid;
        const bool full = row_ok && col + 4 <= cvalid;
        if (row_ok && !full && col < cvalid) continue;  // straddles the end of the row: second pass
        lds_dma<16>(full ? g + (long long)i * gstride + col : zero, m0);
    }
}

// The vector of a tile row that straddles the end of the valid columns (at most one per row): thread `tid`
// of the workgroup loads the one of row `tid` with element loads, and stores it once every tile of the volley
// has been enqueued, so that all these loads are in flight together.  Tiles have at most 256 rows.
struct TileEdge {
    float4 v;
    float *dst;
};

__device__ inline TileEdge tile_edge_load(const float *__restrict__ g, long long gstride, int nrows, int ncols,
                                          int rvalid, int cvalid, float *lds, int pitch, int tid) {
    TileEdge e;
    e.dst = nullptr;
    e.v = make_float4(0.f, 0.f, 0.f, 0.f);
    const int pcol = cvalid & ~3;
    if ((cvalid & 3) && pcol < ncols && tid < nrows && tid < rvalid) {
        const float *src = g + (long long)tid * gstride + pcol;
        e.v.x = src[0];
        if (pcol + 1 < cvalid) e.v.y = src[1];
        if (pcol + 2 < cvalid) e.v.z = src[2];
        e.dst = lds + (size_t)tid * pitch + pcol;
    }
    return e;
}

__device__ inline void tile_edge_store(const TileEdge &e) {
    if (e.dst) *reinterpret_cast<float4 *>(e.dst) = e.v;
}

// ---------------------------------------------------------------------------------------------------------
// Panel product for the projections and their gradients.
//
//   C[n][m] (+)= bias[n] + sum over terms t, samples b (gradient mode) and k of A_t(n,k) * B_t(m,k)
//
// where A_t(n,k) sits at A_t + b*a_s + n*a_n + k*a_k (B alike) and one of the two strides of each operand
// is 1.  The whole 32-row x <=200-deep panel of each operand goes from global memory to LDS in one volley of
// LDS-DMA loads, all in flight together: one trip to memory per panel.  The four waves split the contraction
// in groups of eight k and meet in LDS.  LDS layouts: [k][32 rows] when rows are contiguous in memory
// (fragment = four 4-byte reads, lanes along rows), [row][k] with a pitch of 204 floats (an odd number of
// 16-byte units) when k is (fragment = one 16-byte read); both are free of bank conflicts.
constexpr int PG_KC = 200;          // contraction depth of a panel (multiple of 8)
constexpr int PG_P = PG_KC + 4;     // pitch of the [row][k] layout
constexpr int PG_PANEL = 32 * PG_P; // floats per operand panel (the [k][32] layout needs 32 * PG_KC)

struct PanelArgs {
    const float *A[3], *B[3];  // operands of term t (fan-in) or output o (fan-out)
    float *C[3];
    const float *bias[3];
    const float *zero;         // source of elements that do not exist
    float *part;               // partial sums [nout][groups][N][M] when groups > 1
    int nout, nterm;
    int N, M, K;
    int a_n, a_k, b_m, b_k;
    long long a_s, b_s, c_s;   // per-sample element strides
    int c_n;                   // output row stride (columns contiguous)
    int ns;
    int sum_samples;           // 1: the contraction also runs over the samples (weight gradients)
    int spg, groups;           // samples per workgroup and number of sample groups in that mode
    int accumulate;            // 1: add to what C holds
};

// Panel of rows [r0, r0+32) x k [k0, k0+PG_KC) of an operand with row stride s_r and k stride s_k.
template <bool KMAJ, int NW>
__device__ inline TileEdge panel_load(const float *g, int s_r, int s_k, int r0, int R, int k0, int K, float *lds,
                                      const float *zero, int tid, int wave, int lane) {
    if (KMAJ) {
        const float *t = g + (long long)r0 * s_r + k0;
        tile_dma<NW>(t, s_r, 32, PG_KC, R - r0, K - k0, lds, PG_P, zero, wave, lane);
        return tile_edge_load(t, s_r, 32, PG_KC, R - r0, K - k0, lds, PG_P, tid);
    }
    const float *t = g + (long long)k0 * s_k + r0;
    tile_dma<NW>(t, s_k, PG_KC, 32, K - k0, R - r0, lds, 32, zero, wave, lane);
    return tile_edge_load(t, s_k, PG_KC, 32, K - k0, R - r0, lds, 32, tid);
}

// The four k values [k4, k4+4) of row r.
template <bool KMAJ>
__device__ inline float4 panel_frag(const float *lds, int r, int k4) {
    if (KMAJ) return *reinterpret_cast<const float4 *>(lds + r * PG_P + k4);
    float4 v;
    v.x = lds[k4 * 32 + r];
    v.y = lds[(k4 + 1) * 32 + r];
    v.z = lds[(k4 + 2) * 32 + r];
    v.w = lds[(k4 + 3) * 32 + r];
    return v;
}

__device__ inline void mfma4(mh_f32x16 &acc, const float4 &a, const float4 &b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
}

// NB row blocks of 32 per workgroup share one B panel; each block has its own four waves.  (bx, by, bz): the
// workgroup's place in the product's grid of (column blocks, row blocks, outputs x samples or sample groups).
template <bool A_KMAJ, bool B_KMAJ, int NB>
__device__ __forceinline__ void panel_gemm_body(const PanelArgs &a, unsigned bx, unsigned by, unsigned bz) {
    extern __shared__ __attribute__((aligned(16))) float pg_lds[];
    constexpr int NW = 4 * NB, NT = ATT_NT * NB;
    float *Bs = pg_lds, *As = pg_lds + PG_PANEL;  // As: NB panels
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int nb = wave >> 2, ks = wave & 3;
    const int m0 = (int)bx * 32, n0 = (int)by * (32 * NB);
    int o, b_first, b_count, grp = 0;
    if (a.sum_samples) {
        o = (int)bz / a.groups;
        grp = (int)bz % a.groups;
        b_first = grp * a.spg;
        b_count = min(a.spg, a.ns - b_first);
    } else {
        o = (int)bz / a.ns;
        b_first = (int)bz % a.ns;
        b_count = 1;
    }
    mh_f32x16 acc = {0};
    for (int bi = 0; bi < b_count; ++bi)
        for (int t = 0; t < a.nterm; ++t) {
            const float *Ag = a.A[o * a.nterm + t] + (long long)(b_first + bi) * a.a_s;
            const float *Bg = a.B[o * a.nterm + t] + (long long)(b_first + bi) * a.b_s;
            for (int k0 = 0; k0 < a.K; k0 += PG_KC) {
                __syncthreads();  // the previous panels have been consumed
                TileEdge ea[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    ea[j].dst = nullptr;
                    if (n0 + 32 * j < a.N)
                        ea[j] = panel_load<A_KMAJ, NW>(Ag, a.a_n, a.a_k, n0 + 32 * j, a.N, k0, a.K, As + j * PG_PANEL,
                                                       a.zero, tid, wave, lane);
                }
                const TileEdge eb = panel_load<B_KMAJ, NW>(Bg, a.b_m, a.b_k, m0, a.M, k0, a.K, Bs, a.zero, tid, wave,
                                                           lane);
#pragma unroll
                for (int j = 0; j < NB; ++j) tile_edge_store(ea[j]);
                tile_edge_store(eb);
                wait_vmcnt<0>();
                __syncthreads();
                // groups of eight k (beyond the valid depth the panels hold zeros), dealt to the four waves of a
                // row block in runs; within a group the lower half-wave takes k 0..3 and the upper 4..7
                if (n0 + 32 * nb < a.N) {
                    const float *Aw = As + nb * PG_PANEL;
                    const int ngroups = (min(PG_KC, a.K - k0) + 7) >> 3;
                    const int per = (ngroups + 3) >> 2;
                    const int g_end = min(ngroups, (ks + 1) * per);
                    for (int gq = ks * per; gq < g_end; ++gq) {
                        const int k4 = gq * 8 + half * 4;
                        mfma4(acc, panel_frag<A_KMAJ>(Aw, l32, k4), panel_frag<B_KMAJ>(Bs, l32, k4));
                    }
                }
            }
        }
    __syncthreads();
    float *red = pg_lds;
#pragma unroll
    for (int v = 0; v < 16; ++v) red[(wave * 32 + 8 * (v / 4) + 4 * half + (v % 4)) * ATT_RP + l32] = acc[v];
    __syncthreads();
    const bool partial = a.sum_samples && a.groups > 1;
    float *Cb = partial ? a.part + ((size_t)o * a.groups + grp) * a.N * a.M
                        : a.C[o] + (a.sum_samples ? 0 : (long long)b_first * a.c_s);
    const int c_n = partial ? a.M : a.c_n;
    const float *bias = partial ? nullptr : a.bias[o];
    for (int idx = tid; idx < 1024 * NB; idx += NT) {
        const int n = idx >> 5, m = idx & 31;  // n in [0, 32*NB)
        const float *r = red + ((n >> 5) * 128 + (n & 31)) * ATT_RP + m;
        float v = ((r[0] + r[32 * ATT_RP]) + r[64 * ATT_RP]) + r[96 * ATT_RP];
        if (n0 + n < a.N && m0 + m < a.M) {
            float *dst = Cb + (size_t)(n0 + n) * c_n + m0 + m;
            if (bias) v = v + bias[n0 + n];
            if (a.accumulate && !partial) v = *dst + v;
            *dst = v;
        }
    }
}

template <bool A_KMAJ, bool B_KMAJ, int NB>
__global__ __launch_bounds__(ATT_NT * NB) void panel_gemm_kernel(PanelArgs a) {
    panel_gemm_body<A_KMAJ, B_KMAJ, NB>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Two independent products in one launch (both read what the launch before them wrote, neither reads the other):
// the first n0 workgroups are the first product's grid (gx0 x gy0 x gz0, x fastest), the rest the second's.  The
// block is as large as the larger of the two needs; the waves a product does not use leave at once.
struct PanelPairGrid {
    unsigned n0, gx0, gy0, gx1, gy1;
    int nb0, nb1;
};

template <bool AK0, bool BK0, bool AK1, bool BK1>
__global__ __launch_bounds__(ATT_NT * 2) void panel_gemm_pair_kernel(PanelArgs a, PanelArgs b, PanelPairGrid g) {
    unsigned id = blockIdx.x;
    if (id < g.n0) {
        if ((int)threadIdx.x >= ATT_NT * g.nb0) return;
        const unsigned bx = id % g.gx0, r = id / g.gx0;
        if (g.nb0 == 2)
            panel_gemm_body<AK0, BK0, 2>(a, bx, r % g.gy0, r / g.gy0);
        else
            panel_gemm_body<AK0, BK0, 1>(a, bx, r % g.gy0, r / g.gy0);
    } else {
        id -= g.n0;
        if ((int)threadIdx.x >= ATT_NT * g.nb1) return;
        const unsigned bx = id % g.gx1, r = id / g.gx1;
        if (g.nb1 == 2)
            panel_gemm_body<AK1, BK1, 2>(b, bx, r % g.gy1, r / g.gy1);
        else
            panel_gemm_body<AK1, BK1, 1>(b, bx, r % g.gy1, r / g.gy1);
    }
}

// C_o[i] = sum over groups of part[o][g][i]   (+ what C holds when accumulate)
__device__ __forceinline__ void panel_reduce_body(const PanelArgs &a, int o) {
    const size_t nm = (size_t)a.N * a.M, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nm) return;
    const float *p = a.part + (size_t)o * a.groups * nm + i;
    // eight loads in flight at a time (a serial walk is one trip to memory per group); the sums are added in
    // the order of the groups either way
    float s = 0.f;
    int g = 0;
    for (; g + 8 <= a.groups; g += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[(size_t)(g + j) * nm];
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[j];
    }
    for (; g < a.groups; ++g) s += p[(size_t)g * nm];
    float *dst = a.C[o] + (i / a.M) * a.c_n + (i % a.M);
    *dst = a.accumulate ? *dst + s : s;
}

__global__ __launch_bounds__(256) void panel_reduce_kernel(PanelArgs a) { panel_reduce_body(a, blockIdx.y); }

// ... of two products at once: blockIdx.y runs over the outputs of the first, then of the second
__global__ __launch_bounds__(256) void panel_reduce_pair_kernel(PanelArgs a, PanelArgs b) {
    if ((int)blockIdx.y < a.nout)
        panel_reduce_body(a, blockIdx.y);
    else
        panel_reduce_body(b, (int)blockIdx.y - a.nout);
}

struct AttnArgs {
    const float *q, *k, *v;  // [ns][F][L]
    const float *p;          // probabilities [ns][heads][L][L]   (backward)
    const float *da;         // attention_map gradient [ns][F][L]  (backward)
    const float *dp;         // probability gradient               (backward II)
    const float *rs;         // row sums of dP.P [ns][heads][L]    (backward II)
    float *o0, *o1, *o2;     // kernel outputs (see each kernel)
    const float *zero;       // 256 zero bytes: source of elements that do not exist
    int L, H, heads, F, LP, ns;
    float scale;
    RagDiv d_tiles, d_heads;  // of the kernels up to SQ_L tokens
};

// Forward: o0 = probabilities, o1 = attention_map.  grid (query tiles, heads, samples).
template <int HMAX>
__global__ __launch_bounds__(ATT_NT) void attn_fw_kernel(AttnArgs a) {
    extern __shared__ float att_lds[];
    float *S = att_lds, *vbuf = S + 32 * a.LP, *red = vbuf + HMAX * ATT_VP;
    const int r0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z, L = a.L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t hoff = ((size_t)b * a.F + (size_t)h * a.H) * L;
    scores_to_lds<HMAX>(a.q + hoff, a.k + hoff, L, a.H, r0, a.scale, S, a.LP);
    __syncthreads();
    // softmax of each row over the keys (lib/sources/pulp_act_fp32.c:187-225): max, approximate exponential of
    // the difference, sum, division
    float *P = a.o0 + ((size_t)b * a.heads + h) * L * L;
    for (int row = wave; row < 32; row += 4) {
        float *srow = S + row * a.LP;
        float mx = -FLT_MAX;
        for (int c = lane; c < L; c += 64) mx = fmaxf(mx, srow[c]);
        mx = wave_max(mx);
        float sum = 0.f;
        for (int c = lane; c < L; c += 64) {
            const float e = fastexp_gist(srow[c] - mx);
            srow[c] = e;
            sum += e;
        }
        sum = wave_sum(sum);
        const bool live = r0 + row < L;
        for (int c = lane; c < L; c += 64) {
            const float pv = srow[c] / sum;
            srow[c] = pv;
            if (live) P[(size_t)(r0 + row) * L + c] = pv;
        }
        for (int c = L + lane; c < a.LP - 1; c += 64) srow[c] = 0.f;
    }
    __syncthreads();
    mix_from_lds<HMAX>(a.v + hoff, S, a.LP, L, a.H, r0, a.o1 + hoff, vbuf, red);
}

// Backward, query side: o0 = dP (softmax_buffer gradient), o1 = dq, o2 = row sums of dP.P.
template <int HMAX>
__global__ __launch_bounds__(ATT_NT) void attn_bw_query_kernel(AttnArgs a) {
    extern __shared__ float att_lds[];
    float *S = att_lds, *vbuf = S + 32 * a.LP, *red = vbuf + HMAX * ATT_VP;
    const int r0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z, L = a.L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t hoff = ((size_t)b * a.F + (size_t)h * a.H) * L;
    const size_t poff = ((size_t)b * a.heads + h) * L * L;
    // dP[query][key] = sum_d dA[d][query] v[d][key]   (lib/sources/pulp_mhsa_fp32.c:958-1060)
    scores_to_lds<HMAX>(a.da + hoff, a.v + hoff, L, a.H, r0, 1.0f, S, a.LP);
    __syncthreads();
    // softmax backward (lib/sources/pulp_act_fp32.c:335-390) and the scaling (:1176-1183)
    for (int row = wave; row < 32; row += 4) {
        float *srow = S + row * a.LP;
        const bool live = r0 + row < L;
        const float *prow = a.p + poff + (size_t)(r0 + row) * L;
        float *dprow = a.o0 + poff + (size_t)(r0 + row) * L;
        float sum = 0.f;
        if (live)
            for (int c = lane; c < L; c += 64) sum += srow[c] * prow[c];
        sum = wave_sum(sum);
        for (int c = lane; c < L; c += 64) {
            const float g = srow[c];
            float ds = 0.f;
            if (live) {
                dprow[c] = g;
                ds = ((g - sum) * prow[c]) * a.scale;
            }
            srow[c] = ds;
        }
        for (int c = L + lane; c < a.LP - 1; c += 64) srow[c] = 0.f;
        if (live && lane == 0) a.o2[((size_t)b * a.heads + h) * L + r0 + row] = sum;
    }
    __syncthreads();
    // dq[d][query] = sum_key k[d][key] dS[query][key]   (:1342-1360)
    mix_from_lds<HMAX>(a.k + hoff, S, a.LP, L, a.H, r0, a.o1 + hoff, vbuf, red);
}

// Backward, key side: o0 = dv, o1 = dk for a tile of 32 keys.
//   dv[d][key] = sum_query dA[d][query] P[query][key]                         (:884-902)
//   dk[d][key] = sum_query q[d][query] dS[query][key], dS = (dP - rs) P scale  (:1244-1330)
// dA and q are staged through LDS chunk by chunk of the queries; P and dP are read from global memory with
// the keys on consecutive lanes.
template <int HMAX>
__global__ __launch_bounds__(ATT_NT) void attn_bw_key_kernel(AttnArgs a) {
    extern __shared__ float att_lds[];
    float *abuf = att_lds, *qbuf = abuf + HMAX * ATT_VP, *red = qbuf + HMAX * ATT_VP;
    constexpr int DB = HMAX / 32, KS = 4 / DB;
    constexpr int PER = HMAX * ATT_CK / ATT_NT;
    constexpr int SPW = (ATT_CK / 2) / KS;
    const int c0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z, L = a.L, H = a.H;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int db = wave % DB, ks = wave / DB;
    const size_t hoff = ((size_t)b * a.F + (size_t)h * H) * L;
    const size_t poff = ((size_t)b * a.heads + h) * L * L;
    const float *dA = a.da + hoff, *Q = a.q + hoff, *P = a.p + poff, *dP = a.dp + poff;
    const float *rs = a.rs + ((size_t)b * a.heads + h) * L;
    const int c = c0 + l32;

    float sa[PER], sq[PER], pf[SPW], sf[SPW];
    auto fetch = [&](int q0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + ATT_NT * i, d = idx >> 6, r = q0 + (idx & 63);
            const bool ok = d < H && r < L;
            sa[i] = ok ? dA[(size_t)d * L + r] : 0.f;
            sq[i] = ok ? Q[(size_t)d * L + r] : 0.f;
        }
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const int r = q0 + 2 * (ks * SPW + s) + half;
            const bool ok = r < L && c < L;
            const float pv = ok ? P[(size_t)r * L + c] : 0.f;
            const float g = ok ? dP[(size_t)r * L + c] : 0.f;
            const float rr = ok ? rs[r] : 0.f;
            pf[s] = pv;
            sf[s] = ((g - rr) * pv) * a.scale;
        }
    };
    const int chunks = (L + ATT_CK - 1) / ATT_CK;
    mh_f32x16 accv = {0}, acck = {0};
    fetch(0);
    for (int ch = 0; ch < chunks; ++ch) {
        __syncthreads();
        float pc[SPW], sc[SPW];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = tid + ATT_NT * i;
            abuf[(idx >> 6) * ATT_VP + (idx & 63)] = sa[i];
            qbuf[(idx >> 6) * ATT_VP + (idx & 63)] = sq[i];
        }
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            pc[s] = pf[s];
            sc[s] = sf[s];
        }
        __syncthreads();
        if (ch + 1 < chunks) fetch((ch + 1) * ATT_CK);
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const int kk = 2 * (ks * SPW + s) + half;
            const float av = abuf[(db * 32 + l32) * ATT_VP + kk];
            const float aq = qbuf[(db * 32 + l32) * ATT_VP + kk];
            accv = __builtin_amdgcn_mfma_f32_32x32x2f32(av, pc[s], accv, 0, 0, 0);
            acck = __builtin_amdgcn_mfma_f32_32x32x2f32(aq, sc[s], acck, 0, 0, 0);
        }
    }
    float *outs[2] = {a.o0 + hoff, a.o1 + hoff};
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; ++v)
            red[(wave * 32 + 8 * (v / 4) + 4 * half + (v % 4)) * ATT_RP + l32] = which ? acck[v] : accv[v];
        __syncthreads();
        for (int idx = tid; idx < HMAX * 32; idx += ATT_NT) {
            const int d = idx >> 5, cc = idx & 31;
            float s = 0.f;
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) s += red[((k2 * DB + (d >> 5)) * 32 + (d & 31)) * ATT_RP + cc];
            if (d < H && c0 + cc < L) outs[which][(size_t)d * L + c0 + cc] = s;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// Sequences of at most 256 tokens and heads of at most 64 (HB = 1: 32): the score tile of 32 queries and the one operand
// that a product needs along its other axis are in LDS (the panel): 78 KB for 197 tokens, so that two workgroups share a CU
// and one's loads hide behind the other's products.  32 x 3 heads of 64 and 197 tokens: 37 / 37 / 41 us with all three
// operands resident (150 KB, one workgroup of 16 waves), 30 / 28 / 30 with two workgroups, now 25.7 / 26.0 / 24.6, of which the
// products take 7 / 9 / 7 at the matrix rate.  A workgroup of the forward kernel then took 28 k clocks: 12 until its operands
// were there and multiplied (a CU takes a vector load of 64 lanes every 10 to 20 clocks, whatever its width), 5 of softmax, 4 of
// the value mix, 2 until that was stored.  So what is the same in all lanes is worked out in scalar registers, a wave's four rows
// are reduced side by side, and a head whose [H][L] block starts on 16 bytes and has whole pieces of 16 (LINE) comes in such
// pieces, 50 loads instead of 64 rows of unaligned ones (or of 448 loads of single elements for the scores).
constexpr int SQ_NW = 8;           // waves
constexpr int SQ_NT = SQ_NW * 64;  // threads
constexpr int SQ_RPW = 32 / SQ_NW; // score rows per wave
constexpr int SQ_L = 256;          // tokens
// Pitch of the [d][token] and [row][token] tiles: whole groups of eight and an odd number of 16-byte units, so that
// 16-byte fragments along the tokens meet different banks.
__host__ __device__ constexpr int sq_pitch(int L) { return (L + 7) / 8 * 8 + 4; }
template <int HB>
constexpr size_t sq_lds(int L, bool key) {
    const size_t tiles = (size_t)(32 * HB + (key ? 1 : 32)) * sq_pitch(L), parked = (size_t)SQ_NW * 32 * ATT_RP;
    return (tiles > parked ? tiles : parked) * sizeof(float);
}

static_assert(SQ_RPW == 4 && SQ_L == 256, "the softmax's registers");

// Workgroups go to the eight XCDs in turn, each with an L2 of its own: all tiles of a head take ids of the same XCD, so that
// its operands come from memory once and not once per tile.  False: no head for this workgroup.
struct SqPlace {
    int tile, h, b, part;
};
template <int PARTS>
__device__ inline bool sq_place(const AttnArgs &a, SqPlace &p) {
    const unsigned j = blockIdx.x >> 3, group = rag_quot(j, a.d_tiles), t = j - group * a.d_tiles.d;
    const unsigned head = group * 8u + (blockIdx.x & 7u);
    if (head >= (unsigned)(a.heads * a.ns)) return false;
    p.b = (int)rag_quot(head, a.d_heads);
    p.h = (int)(head - (unsigned)p.b * a.d_heads.d);
    p.tile = (int)(t / (unsigned)PARTS);
    p.part = (int)(t % (unsigned)PARTS);
    return true;
}

// The element `off` bytes behind g, which is the same in all lanes: the load takes it from scalar registers.
__device__ inline float sq_load(const float *g, unsigned off) { return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(g) + off); }
__device__ inline void sq_put(float *g, unsigned off, float v) { *reinterpret_cast<float *>(reinterpret_cast<char *>(g) + off) = v; }

// wave_max and wave_sum of a wave's four rows side by side: one instruction a step and row, its wait states filled by the other
// rows (one after the other, with what the compiler adds for signalling NaNs, 110 more instructions a wave and kernel).
#define SQ_STEP(op, how) op " %0, %0, %0 " how "\n" op " %1, %1, %1 " how "\n" op " %2, %2, %2 " how "\n" op " %3, %3, %3 " how "\n"
#define SQ_ROWS(op)                                                                                                            \
    "s_nop 1\n" SQ_STEP(op, "row_shr:1 row_mask:0xf bank_mask:0xf") SQ_STEP(op, "row_shr:2 row_mask:0xf bank_mask:0xf")         \
        SQ_STEP(op, "row_shr:4 row_mask:0xf bank_mask:0xf") SQ_STEP(op, "row_shr:8 row_mask:0xf bank_mask:0xf")                 \
            SQ_STEP(op, "row_bcast:15 row_mask:0xa bank_mask:0xf") SQ_STEP(op, "row_bcast:31 row_mask:0xc bank_mask:0xf") "s_nop 1"
__device__ inline void sq_max(float (&v)[SQ_RPW]) {
    asm("" SQ_ROWS("v_max_f32_dpp") : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
    for (int i = 0; i < SQ_RPW; ++i) v[i] = last_lane(v[i]);
}
__device__ inline void sq_sum(float (&v)[SQ_RPW]) {
    asm("" SQ_ROWS("v_add_f32_dpp") : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
    for (int i = 0; i < SQ_RPW; ++i) v[i] = last_lane(v[i]);
}

// Rows of V ([H][L]) on their way into the panel: complete once they have been waited for and the edge has been stored, and
// behind a barrier.  LINE: as they lie in memory, a row of L floats behind the other and nothing beyond the last; otherwise at
// sq_pitch(L) with zeros beyond L and H.
template <int HB, bool LINE>
__device__ inline TileEdge sq_fetch(const float *g, int L, int H, float *lds, const float *zero, int tid, int wave, int lane) {
    if (LINE) {
        const int pieces = (H * L) >> 2;  // (in [0, 4096])
        const unsigned to = (unsigned)(uintptr_t)(lds_char *)lds;
        for (int j = wave; j * 64 < pieces; j += SQ_NW)
            if (j * 64 + lane < pieces) lds_dma<16>(g + (j * 64 + lane) * 4, to + (unsigned)j * 1024u);
        return TileEdge{make_float4(0.f, 0.f, 0.f, 0.f), nullptr};
    }
    const int cols = (L + 7) / 8 * 8, col = lane * 4;
    const unsigned to = (unsigned)(uintptr_t)(lds_char *)lds;
    for (int d = wave; d < 32 * HB; d += SQ_NW) {
        const bool full = d < H && col + 4 <= L;
        if (col < cols && (full || d >= H || col >= L)) lds_dma<16>(full ? g + d * L + col : zero, to + (unsigned)(d * sq_pitch(L)) * 4u);
    }
    return tile_edge_load(g, L, 32 * HB, cols, H, L, lds, sq_pitch(L), tid);
}

// S[r][c] = scale * sum_d R[d][r0 + r] * C[d][c] for c < L, zero up to the next group of eight; R and C are [H][L] in
// global memory.  One block of 32 columns per wave.  then(): asks for what the panel holds afterwards; ahead(): for what is
// needed behind the scores.
// LINE: C comes through the panel and R, 32 columns of it, once through LDS; what follows C there arrives during the softmax.
// Otherwise every wave takes both from global memory into registers, which waits for one trip to memory less: forward, us,
// through the panel and straight, 32 x 3 heads of 64 and 197 tokens (LINE) 25.7 and 26.9, 8 x 6 of 32 and 250 (LINE) 13.1 and 13.6,
// 14 x 3 of 64 and 256 22.6 and 21.6, 20 x 4 of 64 and 160 16.6 and 14.6.
template <int HB, bool LINE, typename Then, typename Ahead>
__device__ inline void sq_scores(const float *R, const float *C, int L, int H, int r0, float scale, float *S, float *panel, const float *zero,
                                 int tid, int wave, int lane, Then then, Ahead ahead) {
    constexpr int STEPS = 16 * HB, MINE = STEPS / SQ_NW;
    const int l32 = lane & 31, half = lane >> 5;
    const int pitch = sq_pitch(L), blocks = (L + 31) >> 5;
    static_assert(SQ_L / 32 <= SQ_NW, "a block per wave");
    const int c = wave * 32 + l32;
    const unsigned r = (unsigned)min(r0 + l32, L - 1) * 4u, cc = (unsigned)min(c, L - 1) * 4u, next = half ? (unsigned)L * 4u : 0u;
    auto store = [&](const mh_f32x16 &acc) {
        if (c >= pitch - 4) return;
#pragma unroll
        for (int v = 0; v < 16; ++v) S[(8 * (v / 4) + 4 * half + (v % 4)) * pitch + c] = c < L ? acc[v] * scale : 0.f;
    };
    mh_f32x16 acc = {0};
    if (LINE) {
        float *Rs = pitch >= 32 * HB ? S : panel + 32 * HB * pitch;
        float mine[MINE];
#pragma unroll
        for (int s = 0; s < MINE; ++s) {
            const int d = 2 * (wave + SQ_NW * s);
            mine[s] = sq_load(R + min(d, H - 1) * L, r + (d + 1 < H ? next : 0u));
        }
        sq_fetch<HB, LINE>(C, L, H, panel, zero, tid, wave, lane);
#pragma unroll
        for (int s = 0; s < MINE; ++s) Rs[(2 * (wave + SQ_NW * s) + half) * 32 + l32] = mine[s];
        wait_vmcnt<0>();
        __syncthreads();
        ahead();
        auto form = [&](auto whole) {  // whole: H == 32 HB
            const float *a = Rs + half * 32 + l32, *b = panel + half * L + min(c, L - 1);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const bool in = whole.value || 2 * s + half < H;  // (beyond the head: zeros)
                const float av = a[s * 64], bv = b[2 * s * L];
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? av : 0.f, in ? bv : 0.f, acc, 0, 0, 0);
            }
        };
        if (wave < blocks) {
            if (H == 32 * HB) form(std::true_type{});
            else form(std::false_type{});
        }
        __syncthreads();  // (S takes the place of R, the next panel that of C)
        then();
        if (wave < blocks) store(acc);
    } else {
        auto form = [&](auto whole) {
            float af[STEPS], bf[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int d = whole.value ? 2 * s : min(2 * s, H - 1);
                const unsigned hop = whole.value || 2 * s + 1 < H ? next : 0u;
                af[s] = sq_load(R + d * L, r + hop);
                bf[s] = sq_load(C + d * L, cc + hop);
            }
            __builtin_amdgcn_sched_barrier(0);  // (all of them in flight before the first is waited for)
            then();
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const bool in = whole.value || 2 * s + half < H;
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? af[s] : 0.f, in ? bf[s] : 0.f, acc, 0, 0, 0);
            }
            store(acc);
        };
        if (wave >= blocks) then();
        else if (H == 32 * HB) form(std::true_type{});
        else form(std::false_type{});
        ahead();
    }
    __syncthreads();
}

// Parked partial tiles of the contraction ranges -> out[d][x0 + x] (d < H, x0 + x < L).
template <int HB>
__device__ inline void sq_store(const mh_f32x16 &acc, float *red, int L, int H, int x0, float *__restrict__ out, int tid, int wave,
                                int l32, int half) {
    __syncthreads();  // (the tiles have been read)
#pragma unroll
    for (int v = 0; v < 16; ++v) red[(wave * 32 + 8 * (v / 4) + 4 * half + (v % 4)) * ATT_RP + l32] = acc[v];
    __syncthreads();
    for (int idx = tid; idx < 32 * HB * 32; idx += SQ_NT) {
        const int d = idx >> 5, xx = idx & 31;
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < SQ_NW / HB; ++k) s += red[((HB * k + (d >> 5)) * 32 + (d & 31)) * ATT_RP + xx];
        if (d < H && x0 + xx < L) out[(size_t)d * L + x0 + xx] = s;
    }
}

// V[row][k4 .. k4 + 3] of the panel, zero beyond L.
template <bool LINE>
__device__ inline float4 sq_frag(const float *Vs, int row, int k4, int L, int pitch) {
    if (!LINE) return *reinterpret_cast<const float4 *>(Vs + row * pitch + k4);
    const float *v = Vs + row * L + k4;
    float4 f = make_float4(v[0], v[1], v[2], v[3]);
    if (k4 + 4 > L) {
        f.x = k4 < L ? f.x : 0.f;
        f.y = k4 + 1 < L ? f.y : 0.f;
        f.z = k4 + 2 < L ? f.z : 0.f;
        f.w = 0.f;
    }
    return f;
}

// out[d][r0 + r] = sum_c V[d][c] * S[r][c]: V and S in LDS, both zero beyond L.  Waves: (block of 32 d) x (range of c).
template <int HB, bool LINE>
__device__ inline void sq_mix(const float *Vs, const float *S, int L, int H, int r0, float *__restrict__ out, float *red, int tid,
                              int wave, int l32, int half) {
    constexpr int KS = SQ_NW / HB;
    const int pitch = sq_pitch(L), db = wave % HB, ks = wave / HB;
    const int groups = (L + 7) >> 3, per = (groups + KS - 1) / KS, end = min(groups, (ks + 1) * per);
    mh_f32x16 acc = {0};
    for (int g = ks * per; g < end; ++g) {
        const int k4 = g * 8 + half * 4;
        mfma4(acc, sq_frag<LINE>(Vs, db * 32 + l32, k4, L, pitch), *reinterpret_cast<const float4 *>(S + l32 * pitch + k4));
    }
    sq_store<HB>(acc, red, L, H, r0, out, tid, wave, l32, half);
}

template <int HB, bool LINE>
__global__ __launch_bounds__(SQ_NT, 4) void attn_fw_res_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float att_lds[];
    fetch_args(a);
    SqPlace at;
    if (!sq_place<1>(a, at)) return;
    const int r0 = at.tile * 32, h = at.h, b = at.b, L = a.L, pitch = sq_pitch(L);
    float *S = att_lds, *Vs = S + 32 * pitch;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const size_t hoff = ((size_t)b * a.F + (size_t)h * a.H) * L;
    TileEdge edge;
    sq_scores<HB, LINE>(a.q + hoff, a.k + hoff, L, a.H, r0, a.scale, S, Vs, a.zero, tid, wave, lane,
                        [&] { edge = sq_fetch<HB, LINE>(a.v + hoff, L, a.H, Vs, a.zero, tid, wave, lane); }, [] {});
    // softmax of this wave's rows over the keys (lib/sources/pulp_act_fp32.c:187-225): max, approximate
    // exponential of the difference, sum, division; the rows' reductions run side by side
    float *P = a.o0 + ((size_t)b * a.heads + h) * L * L;
    const int first = wave * SQ_RPW;
    const bool live = r0 + first < L;
    float *rows = S + first * pitch + lane;
    float sv[SQ_RPW][4], mx[SQ_RPW], sum[SQ_RPW] = {};
    if (live) {
#pragma unroll
        for (int i = 0; i < SQ_RPW; ++i) mx[i] = -FLT_MAX;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < L) {
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) mx[i] = fmaxf(mx[i], sv[i][j] = rows[i * pitch + 64 * j]);
            }
        sq_max(mx);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < L) {
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) sum[i] += sv[i][j] = fastexp_below(sv[i][j] - mx[i]);
            }
        sq_sum(sum);
        // (one division for the four rows, in four lanes; the products differ from quotients by an ulp at most)
        float inv = sum[0];
#pragma unroll
        for (int i = 1; i < SQ_RPW; ++i) inv = lane == i ? sum[i] : inv;
        inv = 1.0f / inv;
#pragma unroll
        for (int i = 0; i < SQ_RPW; ++i) sum[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, inv), i));
    }
    tile_edge_store(edge);
    wait_vmcnt<0>();
    if (live) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < L) {
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) {
                    sv[i][j] *= sum[i];
                    rows[i * pitch + 64 * j] = sv[i][j];
                    if (r0 + first + i < L) sq_put(P + (r0 + first + i) * L + 64 * j, (unsigned)lane * 4u, sv[i][j]);
                }
            }
    }
    __syncthreads();
    sq_mix<HB, LINE>(Vs, S, L, a.H, r0, a.o1 + hoff, att_lds, tid, wave, l32, half);
}

template <int HB, bool LINE>
__global__ __launch_bounds__(SQ_NT, 4) void attn_bw_query_res_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float att_lds[];
    fetch_args(a);
    SqPlace at;
    if (!sq_place<1>(a, at)) return;
    const int r0 = at.tile * 32, h = at.h, b = at.b, L = a.L, pitch = sq_pitch(L);
    float *S = att_lds, *Ks = S + 32 * pitch;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const size_t hoff = ((size_t)b * a.F + (size_t)h * a.H) * L;
    const size_t poff = ((size_t)b * a.heads + h) * L * L;
    // dP[query][key] = sum_d dA[d][query] v[d][key]   (lib/sources/pulp_mhsa_fp32.c:958-1060)
    TileEdge edge;
    const int first = wave * SQ_RPW;
    const bool live = r0 + first < L;
    float pr[SQ_RPW][4];  // this wave's probability rows
    sq_scores<HB, LINE>(
        a.da + hoff, a.v + hoff, L, a.H, r0, 1.0f, S, Ks, a.zero, tid, wave, lane,
        [&] {
            if (LINE) {  // (they are waited for here, so that nothing waits for the panel before it is needed)
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) asm volatile("" : "+v"(pr[i][0]), "+v"(pr[i][1]), "+v"(pr[i][2]), "+v"(pr[i][3]));
            }
            edge = sq_fetch<HB, LINE>(a.k + hoff, L, a.H, Ks, a.zero, tid, wave, lane);
        },
        [&] {
            if (!live) return;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (lane + 64 * j < L) {
#pragma unroll
                    for (int i = 0; i < SQ_RPW; ++i) pr[i][j] = sq_load(a.p + poff + min(r0 + first + i, L - 1) * L + 64 * j, (unsigned)lane * 4u);
                }
        });
    // softmax backward (lib/sources/pulp_act_fp32.c:335-390) and the scaling (:1176-1183)
    float *rows = S + first * pitch + lane;
    float gv[SQ_RPW][4], sum[SQ_RPW] = {};
    if (live) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < L) {
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) sum[i] += (gv[i][j] = rows[i * pitch + 64 * j]) * pr[i][j];
            }
        sq_sum(sum);
    }
    tile_edge_store(edge);
    wait_vmcnt<0>();
    if (live) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < L) {
#pragma unroll
                for (int i = 0; i < SQ_RPW; ++i) {
                    if (r0 + first + i < L) sq_put(a.o0 + poff + (r0 + first + i) * L + 64 * j, (unsigned)lane * 4u, gv[i][j]);
                    rows[i * pitch + 64 * j] = ((gv[i][j] - sum[i]) * pr[i][j]) * a.scale;
                }
            }
        if (lane == 0)
#pragma unroll
            for (int i = 0; i < SQ_RPW; ++i)
                if (r0 + first + i < L) a.o2[((size_t)b * a.heads + h) * L + r0 + first + i] = sum[i];
    }
    __syncthreads();
    // dq[d][query] = sum_key k[d][key] dS[query][key]   (:1342-1360)
    sq_mix<HB, LINE>(Ks, S, L, a.H, r0, a.o1 + hoff, att_lds, tid, wave, l32, half);
}

// Key side, a tile of 32 keys: one workgroup forms dv, one dk.  dA (q) is the panel, the key columns of P (and dP) go straight
// to registers, 128 bytes of a query per half wave.  NB: blocks of 32 features a wave forms.  Both (beyond 128 tokens), so that
// no two waves load the same columns: 30 -> 25 us for 32 x 3 heads of 64 and 197 tokens; with fewer tokens an eighth of them is
// a group or two, and one block a wave the better (59 x 3 of 48 and 96 tokens 16.7 against 17.7 us).
//   dv[d][key] = sum_query dA[d][query] P[query][key]                         (:884-902)
//   dk[d][key] = sum_query q[d][query] dS[query][key], dS = (dP - rs) P scale  (:1244-1330)
template <int HB, bool LINE, bool DK, int NB>
__device__ inline void sq_key(const AttnArgs &a, const SqPlace &at, float *lds) {
    constexpr int KS = SQ_NW * NB / HB, PER = 4;  // shares of the queries, groups of eight of them a wave
    const int c0 = at.tile * 32, L = a.L, H = a.H, pitch = sq_pitch(L);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const size_t hoff = ((size_t)at.b * a.F + (size_t)at.h * H) * L, row0 = (size_t)at.b * a.heads + at.h;
    const float *P = a.p + row0 * L * L, *G = a.dp + row0 * L * L;
    const TileEdge edge = sq_fetch<HB, LINE>((DK ? a.q : a.da) + hoff, L, H, lds, a.zero, tid, wave, lane);
    float *rsl = lds + 32 * HB * pitch;  // (zeros up to the next group of eight)
    if (DK && tid < pitch) rsl[tid] = tid < L ? a.rs[row0 * L + tid] : 0.f;
    const int db = NB == 1 ? wave % HB : 0, ks = NB == 1 ? wave / HB : wave;
    const unsigned c = (unsigned)min(c0 + l32, L - 1) * 4u;
    const int groups = (L + 7) >> 3, per = (groups + KS - 1) / KS, g0 = ks * per, end = min(groups, g0 + per);
    tile_edge_store(edge);
    wait_vmcnt<0>();
    __syncthreads();
    float p[PER][4], q[PER][4];  // of the four queries of a group that this half holds
#pragma unroll
    for (int u = 0; u < PER; ++u)
        if (g0 + u < end) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned o = (unsigned)min(((g0 + u) * 8 + j) * L + half * 4 * L, (L - 1) * L) * 4u + c;
                p[u][j] = sq_load(P, o);
                if (DK) q[u][j] = sq_load(G, o);
            }
        }
    __builtin_amdgcn_sched_barrier(0);  // (all of them in flight before the first is waited for)
    mh_f32x16 acc[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) acc[i] = mh_f32x16{0};
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (g0 + u >= end) break;
        const int k4 = (g0 + u) * 8 + half * 4;
        const float4 rs = DK ? *reinterpret_cast<const float4 *>(rsl + k4) : make_float4(0.f, 0.f, 0.f, 0.f);
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = DK ? ((q[u][j] - (j == 0 ? rs.x : j == 1 ? rs.y : j == 2 ? rs.z : rs.w)) * p[u][j]) * a.scale : p[u][j];
        if ((g0 + u) * 8 + 8 > L) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k4 + j >= L) o[j] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) mfma4(acc[i], sq_frag<LINE>(lds, (db + i) * 32 + l32, k4, L, pitch), make_float4(o[0], o[1], o[2], o[3]));
    }
    float *out = (DK ? a.o1 : a.o0) + hoff;
    if (NB == 1) {
        sq_store<HB>(acc[0], lds, L, H, c0, out, tid, wave, l32, half);
    } else {
#pragma unroll
        for (int i = 0; i < NB; ++i) sq_store<1>(acc[i], lds, L, H - 32 * i, c0, out + (size_t)32 * i * L, tid, wave, l32, half);
    }
}

template <int HB, bool LINE>
__global__ __launch_bounds__(SQ_NT, HB == 1 ? 8 : 6) void attn_bw_key_res_kernel(AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float att_lds[];
    fetch_args(a);
    SqPlace at;
    if (!sq_place<2>(a, at)) return;
    if (HB == 2 && a.L > 128) {
        if (at.part == 1) sq_key<HB, LINE, true, HB>(a, at, att_lds);
        else sq_key<HB, LINE, false, HB>(a, at, att_lds);
    } else {
        if (at.part == 1) sq_key<HB, LINE, true, 1>(a, at, att_lds);
        else sq_key<HB, LINE, false, 1>(a, at, att_lds);
    }
}

// Row softmax over H rows of W (one wave per row).
__global__ __launch_bounds__(256) void softmax_fw_rows_kernel(const float *in, float *out, float *maxes,
                                                               float *sums, int H, int W) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= H) return;
    const float *x = in + (size_t)row * W;
    float *y = out + (size_t)row * W;
    float mx = -FLT_MAX;
    for (int c = lane; c < W; c += 64) mx = fmaxf(mx, x[c]);
    mx = wave_max(mx);
    float sum = 0.f;
    for (int c = lane; c < W; c += 64) sum += fastexp_gist(x[c] - mx);
    sum = wave_sum(sum);
    for (int c = lane; c < W; c += 64) y[c] = fastexp_gist(x[c] - mx) / sum;
    if (lane == 0) {
        if (maxes) maxes[row] = mx;
        if (sums) sums[row] = sum;
    }
}

__global__ __launch_bounds__(256) void softmax_bw_rows_kernel(float *in_diff, const float *out, const float *out_diff,
                                                               float *sums, int H, int W) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= H) return;
    const float *y = out + (size_t)row * W, *g = out_diff + (size_t)row * W;
    float sum = 0.f;
    for (int c = lane; c < W; c += 64) sum += g[c] * y[c];
    sum = wave_sum(sum);
    for (int c = lane; c < W; c += 64) in_diff[(size_t)row * W + c] = (g[c] - sum) * y[c];
    if (lane == 0 && sums) sums[row] = sum;
}

// ---------------------------------------------------------------------------------------------------------

struct MhsaDims {
    int L, E, F, heads, H;
};

static int mhsa_dims(const Mhsa_args *a, MhsaDims &m, const char *fn, bool backward) {
    auto bad = [&](const char *what) {
        printf("[%s] %s\n", fn, what);
        set_error("%s: %s", fn, what);
        return 1;
    };
    if (!a || !a->input || !a->output || !a->coeff_in_q || !a->coeff_in_k || !a->coeff_in_v || !a->coeff_out ||
        !a->q || !a->k || !a->v || !a->attention_map || !a->softmax_buffer)
        return bad("null argument structure");
    m.L = a->input->H;
    m.E = a->input->W;
    m.F = a->attention_map->W;
    m.heads = a->n_heads;
    if (m.L <= 0 || m.E <= 0 || m.F <= 0 || m.heads <= 0 || m.F % m.heads) return bad("invalid attention geometry");
    m.H = m.F / m.heads;
    if (m.H > 128) return bad("head size above 128 is not supported");
    if (m.L > 1024) return bad("sequence length above 1024 is not supported");
    const struct blob *act[] = {a->input, a->output, a->q, a->k, a->v, a->attention_map, a->softmax_buffer};
    for (const struct blob *bl : act)
        if (!bl->data || (backward && !bl->diff)) return bad("null activation buffer");
    const struct blob *wts[] = {a->coeff_in_q, a->coeff_in_k, a->coeff_in_v, a->coeff_out};
    for (const struct blob *bl : wts)
        if (!bl->data || (backward && !bl->diff)) return bad("null weight buffer");
    return 0;
}

static int att_lp(int L) { return ((L + ATT_CK - 1) / ATT_CK) * ATT_CK + 1; }

template <int HMAX>
static int launch_attn(int which, AttnArgs &a, int ns) {
    const size_t tile = (size_t)32 * a.LP, stage = (size_t)HMAX * ATT_VP, red = (size_t)4 * 32 * ATT_RP;
    const size_t lds = (which == 2 ? 2 * stage + red : tile + stage + red) * sizeof(float);
    void (*kern)(AttnArgs) =
        which == 0 ? attn_fw_kernel<HMAX> : which == 1 ? attn_bw_query_kernel<HMAX> : attn_bw_key_kernel<HMAX>;
    if (lds > 150 * 1024) {
        set_error("attention tile needs %zu bytes of LDS", lds);
        return 1;
    }
    static bool attr_set[3] = {false, false, false};
    if (!attr_set[which]) {
        if (!hip_ok(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024),
                    "hipFuncSetAttribute"))
            return 2;
        attr_set[which] = true;
    }
    dim3 grid((a.L + 31) / 32, a.heads, ns);
    hipLaunchKernelGGL(kern, grid, dim3(ATT_NT), lds, state().stream, a);
    return hip_ok(hipGetLastError(), "attention launch") ? 0 : 2;
}

template <int HB, bool LINE>
static int launch_attn_res(int which, AttnArgs &a, int ns) {
    void (*kern)(AttnArgs) = which == 0 ? attn_fw_res_kernel<HB, LINE> : which == 1 ? attn_bw_query_res_kernel<HB, LINE> : attn_bw_key_res_kernel<HB, LINE>;
    static bool attr_set[3] = {false, false, false};
    if (!attr_set[which]) {
        if (!hip_ok(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)sq_lds<HB>(SQ_L, which == 2)),
                    "hipFuncSetAttribute"))
            return 2;
        attr_set[which] = true;
    }
    a.ns = ns;
    a.d_tiles = rag_div((long long)((a.L + 31) / 32) * (which == 2 ? 2 : 1));
    a.d_heads = rag_div(a.heads);
    const long long blocks = ((long long)ns * a.heads + 7) / 8 * 8 * ((a.L + 31) / 32) * (which == 2 ? 2 : 1);
    if (blocks >= (1ll << 31)) {
        set_error("attention: too many heads");
        return 1;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(SQ_NT), sq_lds<HB>(a.L, which == 2), state().stream, a);
    return hip_ok(hipGetLastError(), "attention launch") ? 0 : 2;
}

static int launch_attn_any(int which, AttnArgs &a, int ns) {
    if (a.L <= SQ_L && a.H <= 64) {
        a.zero = static_cast<const float *>(state().zeros);
        if (!a.zero) return 2;
        // LINE: every head's block in whole pieces of 16 bytes.  Rows of whole pieces (L % 4 == 0) would meet few banks that way.
        const uintptr_t at = reinterpret_cast<uintptr_t>(which == 2 ? a.q : a.k) | reinterpret_cast<uintptr_t>(which == 2 ? a.da : a.v);
        if (a.L % 4 && a.H % 4 == 0 && at % 16 == 0) return a.H <= 32 ? launch_attn_res<1, true>(which, a, ns) : launch_attn_res<2, true>(which, a, ns);
        return a.H <= 32 ? launch_attn_res<1, false>(which, a, ns) : launch_attn_res<2, false>(which, a, ns);
    }
    if (a.H <= 32) return launch_attn<32>(which, a, ns);
    if (a.H <= 64) return launch_attn<64>(which, a, ns);
    return launch_attn<128>(which, a, ns);
}

// Sample groups the gradient mode of the panel product uses for `nout` N x M outputs: enough workgroups to
// fill the chip a few times over.
static int panel_groups(int nout, int N, int M, int ns) {
    const long tiles = (long)((N + 31) / 32) * ((M + 31) / 32) * nout;
    long groups = (4L * state().num_cu + tiles - 1) / tiles;
    if (groups > ns) groups = ns;
    return groups < 1 ? 1 : (int)groups;
}

static size_t panel_part_floats(int nout, int N, int M, int ns) {
    const int g = panel_groups(nout, N, M, ns);
    return g > 1 ? (size_t)nout * g * N * M : 0;
}

// Launches the panel product; `p` carries operands, strides and sizes, this fills in the rest.  In gradient
// mode (sum_samples) the partial sums of the sample groups go to `part` and a second kernel adds them.
// What a launch of the panel product needs besides its arguments.
struct PanelPlan {
    bool ak, bk;
    int nb;
    dim3 grid;
    size_t lds;
};

// Fills in the fields of `p` the caller leaves open (zero page, sample groups, partial sums) and works out the
// launch.  0, or the error code.
static int panel_plan(PanelArgs &p, float *part, PanelPlan &pl) {
    State &st = state();
    p.zero = static_cast<const float *>(st.zeros);
    if (!p.zero) return 2;
    if ((p.a_k != 1 && p.a_n != 1) || (p.b_k != 1 && p.b_m != 1)) {
        set_error("panel product: operand without a unit stride");
        return 1;
    }
    pl.ak = p.a_k == 1;
    pl.bk = p.b_k == 1;
    p.groups = 1;
    p.spg = p.ns;
    p.part = nullptr;
    if (p.sum_samples) {
        const int groups = panel_groups(p.nout, p.N, p.M, p.ns);
        if (groups > 1) {
            p.spg = (p.ns + groups - 1) / groups;
            p.groups = (p.ns + p.spg - 1) / p.spg;
            p.part = part;
            if (!part) return 2;
        }
    }
    // Two row blocks per workgroup (the B panel is fetched once for both) when single blocks would already
    // queue up behind each other on the CUs.
    const size_t zdim = p.sum_samples ? (size_t)p.nout * p.groups : (size_t)p.nout * p.ns;
    const size_t single = (size_t)((p.M + 31) / 32) * ((p.N + 31) / 32) * zdim;
    pl.nb = (p.N > 32 && single > (size_t)3 * st.num_cu) ? 2 : 1;
    pl.lds = (size_t)(1 + pl.nb) * PG_PANEL * sizeof(float);  // 52 KB or 78 KB
    pl.grid = dim3((p.M + 31) / 32, (p.N + 32 * pl.nb - 1) / (32 * pl.nb), (unsigned)zdim);
    if (pl.grid.y > 65535u || zdim > 65535u) {
        set_error("panel product: grid too large");
        return 1;
    }
    return 0;
}

static int launch_panel_reduce(PanelArgs &p) {
    if (p.groups <= 1) return 0;
    hipLaunchKernelGGL(panel_reduce_kernel, dim3((unsigned)(((size_t)p.N * p.M + 255) / 256), p.nout), dim3(256), 0,
                       state().stream, p);
    p.groups = 0;  // (added up: a later call finds nothing to do)
    return hip_ok(hipGetLastError(), "panel reduce launch") ? 0 : 2;
}

// The additions of two products' sample groups in one launch.
static int launch_panel_reduce_pair(PanelArgs &p0, PanelArgs &p1) {
    if (p0.groups <= 1) return launch_panel_reduce(p1);
    if (p1.groups <= 1) return launch_panel_reduce(p0);
    const size_t nm0 = (size_t)p0.N * p0.M, nm1 = (size_t)p1.N * p1.M, nm = nm0 > nm1 ? nm0 : nm1;
    hipLaunchKernelGGL(panel_reduce_pair_kernel, dim3((unsigned)((nm + 255) / 256), p0.nout + p1.nout), dim3(256), 0,
                       state().stream, p0, p1);
    p0.groups = p1.groups = 0;
    return hip_ok(hipGetLastError(), "panel reduce launch") ? 0 : 2;
}

// Launches the panel product; `p` carries operands, strides and sizes, this fills in the rest.  In gradient
// mode (sum_samples) the partial sums of the sample groups go to `part` and a second kernel adds them.
static int launch_panel(PanelArgs &p, float *part) {
    State &st = state();
    PanelPlan pl;
    if (int rc = panel_plan(p, part, pl)) return rc;
    const bool ak = pl.ak, bk = pl.bk;
    void (*kern)(PanelArgs);
    if (pl.nb == 2)
        kern = ak ? (bk ? panel_gemm_kernel<true, true, 2> : panel_gemm_kernel<true, false, 2>)
                  : (bk ? panel_gemm_kernel<false, true, 2> : panel_gemm_kernel<false, false, 2>);
    else
        kern = ak ? (bk ? panel_gemm_kernel<true, true, 1> : panel_gemm_kernel<true, false, 1>)
                  : (bk ? panel_gemm_kernel<false, true, 1> : panel_gemm_kernel<false, false, 1>);
    if (pl.nb == 2) {
        static bool attr_set[4] = {false, false, false, false};
        const int which = (ak ? 2 : 0) + (bk ? 1 : 0);
        if (!attr_set[which]) {
            if (!hip_ok(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds),
                        "hipFuncSetAttribute"))
                return 2;
            attr_set[which] = true;
        }
    }
    hipLaunchKernelGGL(kern, pl.grid, dim3(ATT_NT * pl.nb), pl.lds, st.stream, p);
    if (!hip_ok(hipGetLastError(), "panel product launch")) return 2;
    return launch_panel_reduce(p);
}

// Two independent panel products in one launch (the two the backward pass has twice: the gradient of the output
// weights with the gradient of the attention map, and the gradients of the input weights with the gradient of the
// input), each followed by the addition of its sample groups where it has any.  `PAIR` names the orientations.
template <bool AK0, bool BK0, bool AK1, bool BK1>
static int launch_panel_pair(PanelArgs &p0, float *part0, PanelArgs &p1, float *part1, bool add_now = true) {
    State &st = state();
    PanelPlan l0, l1;
    if (int rc = panel_plan(p0, part0, l0)) return rc;
    if (int rc = panel_plan(p1, part1, l1)) return rc;
    const size_t n0 = (size_t)l0.grid.x * l0.grid.y * l0.grid.z, n1 = (size_t)l1.grid.x * l1.grid.y * l1.grid.z;
    if (l0.ak != AK0 || l0.bk != BK0 || l1.ak != AK1 || l1.bk != BK1 || n0 + n1 >= ((size_t)1 << 31) ||
        st.gemm_path == 7) {  // (not this pair, or one product at a time asked for)
        if (int rc = launch_panel(p0, part0)) return rc;
        return launch_panel(p1, part1);
    }
    void (*kern)(PanelArgs, PanelArgs, PanelPairGrid) = panel_gemm_pair_kernel<AK0, BK0, AK1, BK1>;
    const size_t lds = l0.lds > l1.lds ? l0.lds : l1.lds;
    static bool attr_set = false;
    if (!attr_set) {
        if (!hip_ok(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)(3 * PG_PANEL * sizeof(float))),
                    "hipFuncSetAttribute"))
            return 2;
        attr_set = true;
    }
    PanelPairGrid g;
    g.n0 = (unsigned)n0;
    g.gx0 = l0.grid.x; g.gy0 = l0.grid.y;
    g.gx1 = l1.grid.x; g.gy1 = l1.grid.y;
    g.nb0 = l0.nb; g.nb1 = l1.nb;
    const int nbmax = l0.nb > l1.nb ? l0.nb : l1.nb;
    hipLaunchKernelGGL(kern, dim3((unsigned)(n0 + n1)), dim3(ATT_NT * nbmax), lds, st.stream, p0, p1, g);
    if (!hip_ok(hipGetLastError(), "panel product pair launch")) return 2;
    return add_now ? launch_panel_reduce_pair(p0, p1) : 0;  // (else the caller adds the groups up later)
}

// out[b][N x L] = Wt(N x K) . act[b][K x L]: a weight matrix with element (n,k) at n*a_n + k*a_k against a
// batch of activations (tokens contiguous).
static PanelArgs weights_times_acts(int N, int K, int L, int ns, int a_n, int a_k) {
    PanelArgs p = {};
    p.nout = p.nterm = 1;
    p.N = N;
    p.M = L;
    p.K = K;
    p.a_n = a_n;
    p.a_k = a_k;
    p.b_m = 1;
    p.b_k = L;
    p.b_s = (long long)K * L;
    p.c_s = (long long)N * L;
    p.c_n = L;
    p.ns = ns;
    return p;
}

// out[N x M] = sum over samples and tokens of A[b][N x L] . B[b][M x L]^T  (weight gradients).
static PanelArgs acts_times_acts(int N, int M, int L, int ns) {
    PanelArgs p = {};
    p.nout = p.nterm = 1;
    p.N = N;
    p.M = M;
    p.K = L;
    p.a_n = L;
    p.a_k = 1;
    p.a_s = (long long)N * L;
    p.b_m = L;
    p.b_k = 1;
    p.b_s = (long long)M * L;
    p.c_n = M;
    p.ns = ns;
    p.sum_samples = 1;
    return p;
}

// The same products for the kernel of any size and alignment: out[b][N x L] = W(N x K) . act[b][K x L] (tiles stay inside a
// sample), W with rows of K or, transposed, columns of N; and out[N x M] = sum over samples and tokens.  Activations are
// formed in one tile shape with the contraction whole, so that a sample's do not depend on the batch it is in.
static RagOp rag_matrix(const float *p, int rows, int row_stride, int k_stride, long long run = 0, long long outer = 0) {
    RagOp o = {};
    o.p = reinterpret_cast<const char *>(p);
    o.rows = rows;
    o.row_b = (unsigned)row_stride * 4u;
    o.k_b = (unsigned)k_stride * 4u;
    o.run_b = run * 4;
    o.outer_b = outer * 4;
    return o;
}
static RagProd rag_weights_times_acts(const float *W, bool transposed, const float *act, float *out, int N, int K, int L, int ns) {
    RagProd p = {};
    p.a = transposed ? rag_matrix(W, N, 1, N) : rag_matrix(W, N, K, 1);
    p.b = rag_matrix(act, L, 1, L, 0, (long long)K * L);
    p.C = out;
    p.N = N;
    p.M = ns * L;
    p.m_in = L;
    p.outer = ns;
    p.K = K;
    p.runs = 1;
    p.cn = rag_axis(N, L);
    p.cm = rag_axis2(L, 1, N * L);
    p.whole_k = 1;
    return p;
}
static RagProd rag_acts_times_acts(const float *A, const float *B, float *out, int N, int M, int L, int ns) {
    RagProd p = {};
    p.a = rag_matrix(A, N, L, 1, (long long)N * L);
    p.b = rag_matrix(B, M, L, 1, (long long)M * L);
    p.C = out;
    p.N = N;
    p.M = p.m_in = M;
    p.outer = 1;
    p.K = L;
    p.runs = ns;
    p.cn = rag_axis(N, M);
    p.cm = rag_axis(M, 1);
    return p;
}
// (small tiles with all waves on the contraction up to 128 tokens: 92 -> 65 us for 7 x 19 tokens, 125 -> 96 for 8 x 64)
static int rag_tile_of(int L) { return L <= 128 ? 32 : 64; }
// Rows and runs of k hold whole pieces (the panels take what has shorter ones, and what paths 6 and 7 ask of them).  Against
// the panels: 83 -> 65 us for 7 x 6 heads of 48 and 19 tokens, 507 -> 430 for 46 x 6 and 192, 123 -> 96 for 8 x 8 of 64 and 64
// tokens, 222 -> 195 for 32 x 3 of 64 and 197, all forward + backward.  Single samples of up to some hundred tokens would be
// faster there (61.7 against 73.0 us for 3 heads of 64 and 197 tokens), but a sample's results are the same bits in every
// batch, so that both cannot be had.
static bool rag_takes(const MhsaDims &m) {
    const int path = state().gemm_path;
    return path != 6 && path != 7 && m.L >= 4 && m.E >= 4 && m.F >= 4 && m.L < (1 << 20) && m.E < (1 << 20) && m.F < (1 << 20);
}

static bool mhsa_fits(const MhsaDims &m, int ns) {
    const size_t lim = (size_t)1 << 31;
    return (size_t)ns * m.E * m.L < lim && (size_t)ns * m.F * m.L < lim && (size_t)ns * m.heads * m.L * m.L < lim &&
           (size_t)m.E * m.F < lim;
}

static int mhsa_fw(const Mhsa_args *a, int ns, const char *fn) {
    MhsaDims m;
    if (int rc = mhsa_dims(a, m, fn, false)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    if (!mhsa_fits(m, ns)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    state().last_gemm_form = 0;
    const int L = m.L, E = m.E, F = m.F;
    const size_t xe = (size_t)ns * E * L, fe = (size_t)ns * F * L, pe = (size_t)ns * m.heads * L * L;
    Stager sg;
    const float *X = sg.in(a->input->data, xe);
    const struct blob *wb[3] = {a->coeff_in_q, a->coeff_in_k, a->coeff_in_v};
    const struct blob *bb[3] = {a->bias_in_q, a->bias_in_k, a->bias_in_v};
    struct blob *ob[3] = {a->q, a->k, a->v};
    const float *W[3], *bias[3];
    float *QKV[3];
    for (int j = 0; j < 3; ++j) {
        W[j] = sg.in(wb[j]->data, (size_t)E * F);
        bias[j] = (bb[j] && bb[j]->data) ? sg.in(bb[j]->data, (size_t)F) : nullptr;
        QKV[j] = sg.out(ob[j]->data, fe);
    }
    const float *Wo = sg.in(a->coeff_out->data, (size_t)E * F);
    float *att = sg.out(a->attention_map->data, fe);
    float *P = sg.out(a->softmax_buffer->data, pe);
    float *Y = sg.out(a->output->data, xe);
    if (sg.failed()) return 2;
    int rc = 0;
    const bool rag = rag_takes(m);
    if (rag) {
        RagArgs r = {};
        r.shape = rag_tile_of(L);
        r.count = 3;
        for (int j = 0; j < 3; ++j) {
            r.p[j] = rag_weights_times_acts(W[j], true, X, QKV[j], F, E, L, ns);
            r.p[j].bias = bias[j];
            r.p[j].bias_n = 1;
        }
        rc = ragged<float>(r, RAG_RC, RAG_RC, RAG_RC, RAG_RC);
    } else {
        // q/k/v[F x L] = W^T . X + bias in one launch (weights stored E x F: lib/sources/pulp_mhsa_fp32.c:70-325)
        PanelArgs p = weights_times_acts(F, E, L, ns, 1, F);
        p.nout = 3;
        for (int j = 0; j < 3; ++j) {
            p.A[j] = W[j];
            p.B[j] = X;
            p.C[j] = QKV[j];
            p.bias[j] = bias[j];
        }
        rc = launch_panel(p, nullptr);
    }
    if (rc == 0) {
        AttnArgs t = {};
        t.q = QKV[0];
        t.k = QKV[1];
        t.v = QKV[2];
        t.o0 = P;
        t.o1 = att;
        t.L = L;
        t.H = m.H;
        t.heads = m.heads;
        t.F = F;
        t.LP = att_lp(L);
        t.scale = q_rsqrt_host((float)m.H);
        rc = launch_attn_any(0, t, ns);
    }
    if (rc == 0 && rag) {
        RagArgs r = {};
        r.shape = rag_tile_of(L);
        r.count = 1;
        r.p[0] = rag_weights_times_acts(Wo, false, att, Y, E, F, L, ns);
        rc = ragged<float>(r, RAG_KC, RAG_RC, RAG_KC, RAG_RC);
    } else if (rc == 0) {
        // output[E x L] = Wout[E x F] . attention_map (:599-609)
        PanelArgs p = weights_times_acts(E, F, L, ns, F, 1);
        p.A[0] = Wo;
        p.B[0] = att;
        p.C[0] = Y;
        rc = launch_panel(p, nullptr);
    }
    return sg.finish(rc);
}

static int mhsa_bw(const Mhsa_args *a, int ns, const char *fn) {
    MhsaDims m;
    if (int rc = mhsa_dims(a, m, fn, true)) return rc;
    if (ns <= 0) return 0;
    if (!ensure_init()) return 2;
    if (!mhsa_fits(m, ns)) {
        set_error("%s: tensor larger than 2^31 elements", fn);
        return 1;
    }
    const int L = m.L, E = m.E, F = m.F;
    const size_t xe = (size_t)ns * E * L, fe = (size_t)ns * F * L, pe = (size_t)ns * m.heads * L * L;
    const size_t rows = (size_t)ns * m.heads * L;
    Stager sg;
    const float *X = sg.in(a->input->data, xe);
    const float *dY = sg.in(a->output->diff, xe);
    float *dX = sg.inout(a->input->diff, xe);
    const struct blob *wb[3] = {a->coeff_in_q, a->coeff_in_k, a->coeff_in_v};
    struct blob *ob[3] = {a->q, a->k, a->v};
    const float *W[3], *QKV[3];
    float *dW[3], *dQKV[3];
    for (int j = 0; j < 3; ++j) {
        W[j] = sg.in(wb[j]->data, (size_t)E * F);
        dW[j] = sg.out(wb[j]->diff, (size_t)E * F);
        QKV[j] = sg.in(ob[j]->data, fe);
        dQKV[j] = sg.out(ob[j]->diff, fe);
    }
    const float *Wo = sg.in(a->coeff_out->data, (size_t)E * F);
    float *dWo = sg.out(a->coeff_out->diff, (size_t)E * F);
    const float *att = sg.in(a->attention_map->data, fe);
    float *datt = sg.out(a->attention_map->diff, fe);
    const float *P = sg.in(a->softmax_buffer->data, pe);
    float *dP = sg.out(a->softmax_buffer->diff, pe);
    if (sg.failed()) return 2;
    const bool rag = rag_takes(m);  // (its partial sums, where there are any, are in the workspace)
    state().last_gemm_form = 0;
    const size_t p1 = rag ? 0 : panel_part_floats(1, E, F, ns), p3 = rag ? 0 : panel_part_floats(3, F, E, ns);
    float *rs = static_cast<float *>(scratch((rows + p1 + p3) * sizeof(float)));
    if (!rs) return 2;
    float *part_o = rs + rows, *part_i = part_o + p1;  // sample-group sums of the output / the input weights' gradients
    int rc = 0;
    // dWout[E x F] = sum over samples of dY . att^T (:742-760) and datt[F x L] = Wout^T . dY (:816-834), one launch;
    // the sample groups of dWout are added up at the end, together with those of the input weights' gradients
    PanelArgs pwo = acts_times_acts(E, F, L, ns);
    if (rag) {  // (dWout comes with the other weights' gradients)
        RagArgs r = {};
        r.shape = rag_tile_of(L);
        r.count = 1;
        r.p[0] = rag_weights_times_acts(Wo, true, dY, datt, F, E, L, ns);
        rc = ragged<float>(r, RAG_RC, RAG_RC, RAG_RC, RAG_RC);
    } else {
        pwo.A[0] = dY;
        pwo.B[0] = att;
        pwo.C[0] = dWo;
        PanelArgs q = weights_times_acts(F, E, L, ns, 1, F);
        q.A[0] = Wo;
        q.B[0] = dY;
        q.C[0] = datt;
        rc = launch_panel_pair<true, true, false, false>(pwo, part_o, q, nullptr, false);
    }
    AttnArgs t = {};
    t.q = QKV[0];
    t.k = QKV[1];
    t.v = QKV[2];
    t.p = P;
    t.da = datt;
    t.L = L;
    t.H = m.H;
    t.heads = m.heads;
    t.F = F;
    t.LP = att_lp(L);
    t.scale = q_rsqrt_host((float)m.H);
    if (rc == 0) {
        t.o0 = dP;
        t.o1 = dQKV[0];
        t.o2 = rs;
        rc = launch_attn_any(1, t, ns);
    }
    if (rc == 0) {
        t.dp = dP;
        t.rs = rs;
        t.o0 = dQKV[2];
        t.o1 = dQKV[1];
        t.o2 = nullptr;
        rc = launch_attn_any(2, t, ns);
    }
    if (rc == 0 && rag) {
        RagArgs r = {};
        r.shape = rag_tile_of(L);
        r.count = 5;
        RagProd &x = r.p[0];
        x = rag_weights_times_acts(W[0], false, dQKV[0], dX, E, F, L, ns);
        x.runs = 3;
        x.add = 1;
        for (int j = 0; j < 2; ++j) {
            r.hop_a[j] = reinterpret_cast<const char *>(W[j + 1]) - reinterpret_cast<const char *>(W[j]);
            r.hop_b[j] = reinterpret_cast<const char *>(dQKV[j + 1]) - reinterpret_cast<const char *>(dQKV[j]);
        }
        for (int j = 0; j < 3; ++j) r.p[1 + j] = rag_acts_times_acts(dQKV[j], X, dW[j], F, E, L, ns);
        r.p[4] = rag_acts_times_acts(dY, att, dWo, E, F, L, ns);
        rc = ragged<float>(r, RAG_KC, RAG_RC, RAG_KC, RAG_KC);
    } else if (rc == 0) {
        // dW_{q,k,v}[F x E] = sum over samples of d{q,k,v} . X^T (:1425-1560) and
        // dX[E x L] += W_q . dq + W_k . dk + W_v . dv (:1589-1745), one launch
        PanelArgs p = acts_times_acts(F, E, L, ns);
        p.nout = 3;
        for (int j = 0; j < 3; ++j) {
            p.A[j] = dQKV[j];
            p.B[j] = X;
            p.C[j] = dW[j];
        }
        PanelArgs q = weights_times_acts(E, F, L, ns, F, 1);
        q.nterm = 3;
        for (int j = 0; j < 3; ++j) {
            q.A[j] = W[j];
            q.B[j] = dQKV[j];
        }
        q.C[0] = dX;
        q.accumulate = 1;
        rc = launch_panel_pair<true, true, true, false>(p, part_i, q, nullptr, false);
        if (rc == 0) rc = launch_panel_reduce_pair(pwo, p);
    }
    return sg.finish(rc);
}

static int softmax_rows(const softmax_args *a, bool backward, const char *fn) {
    if (!a || a->H <= 0 || a->W <= 0 || !a->output_data || (backward ? (!a->input_diff || !a->output_diff)
                                                                      : !a->input_data)) {
        printf("[%s] invalid arguments\n", fn);
        set_error("%s: invalid arguments", fn);
        return 1;
    }
    if (!ensure_init()) return 2;
    const size_t n = (size_t)a->H * a->W;
    Stager sg;
    dim3 grid((a->H + 3) / 4);
    if (!backward) {
        // the rows may be transformed in place (input == output): every element is read and written by one lane
        const float *in;
        float *out;
        if (a->output_data == a->input_data) {
            out = sg.inout(a->output_data, n);
            in = out;
        } else {
            in = sg.in(a->input_data, n);
            out = sg.out(a->output_data, n);
        }
        float *mx = a->maxes ? sg.out(a->maxes, (size_t)a->H) : nullptr;
        float *sm = a->sums ? sg.out(a->sums, (size_t)a->H) : nullptr;
        if (sg.failed()) return 2;
        hipLaunchKernelGGL(softmax_fw_rows_kernel, grid, dim3(256), 0, state().stream, in, out, mx, sm, a->H, a->W);
    } else {
        const float *y = sg.in(a->output_data, n);
        const float *g = sg.in(a->output_diff, n);
        float *gi = sg.out(a->input_diff, n);
        float *sm = a->sums ? sg.out(a->sums, (size_t)a->H) : nullptr;
        if (sg.failed()) return 2;
        hipLaunchKernelGGL(softmax_bw_rows_kernel, grid, dim3(256), 0, state().stream, gi, y, g, sm, a->H, a->W);
    }
    return sg.finish(hip_ok(hipGetLastError(), "softmax launch") ? 0 : 2);
}

}  // namespace ptl

extern "C" {

int ptl_mhsa_fp32_fw_batched(const struct Mhsa_args *a, int nsamples) {
    return ptl::mhsa_fw(a, nsamples, "pulp_mhsa_fp32_fw_cl");
}
int ptl_mhsa_fp32_bw_batched(const struct Mhsa_args *a, int nsamples) {
    return ptl::mhsa_bw(a, nsamples, "pulp_mhsa_fp32_bw_cl");
}
int ptl_internal_softmax_fp32(const struct softmax_args *a, int backward) {
    return ptl::softmax_rows(a, backward != 0, backward ? "pulp_softmax_fp32_bw_cl" : "pulp_softmax_fp32_fw_cl");
}

}  // extern "C"
