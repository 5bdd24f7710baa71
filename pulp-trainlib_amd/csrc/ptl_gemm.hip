// MFMA GEMM over separable index maps: C(n,m) = sum_k A(n,k) * B(m,k).
//
// One kernel family serves every GEMM-shaped step of the training core.  The
// two operands are described by separable index maps (ptl_common.hpp), so the
// implicit im2col gathers of Conv2D forward / weight-gradient / input-gradient,
// the batched pointwise and Linear products and the plain mm() contract are
// all the same code: only the maps differ.  Patch matrices are never
// materialised; patch elements are gathered from the tensor into the LDS tile.
//
// Work decomposition (gfx950, 64-wide waves):
//   * workgroup = 256 threads = 4 waves, computes a BM x BN tile of C;
//   * k is consumed in slabs of 64 bytes per row (32 halves or 16 floats),
//     staged global -> registers -> LDS with two LDS buffers, one barrier per
//     slab; LDS rows are k-contiguous with an 80-byte pitch so every MFMA
//     operand fragment is one 16-byte LDS read;
//   * fp16: v_mfma_f32_32x32x16_f16 (fp32 accumulate); fp32: v_mfma_f32_32x32x2_f32;
//   * optional split-K: grid.y slices k, fp32 partials go to a workspace and a
//     second kernel sums them in a fixed order (deterministic).
#include "ptl_common.hpp"
#include "ptl_ragged.hpp"
#include "ptl_sum.hpp"
#include "ptl_gemm_async.hpp"

#include <algorithm>

namespace ptl {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T>
struct Traits;
template <>
struct Traits<float> {
    static constexpr int VEC = 4;   // elements per 16-byte vector
    static constexpr int BKE = 16;  // elements of k per slab
};
template <>
struct Traits<half_t> {
    static constexpr int VEC = 8;
    static constexpr int BKE = 32;
};

constexpr int PITCH = 80;      // bytes per LDS tile row: 64 data + 16 pad
constexpr int KW = 512;        // k indices decoded per look-up window
constexpr int HW_BIAS = 8192;  // coordinate bias of packed look-up entries

// Look-up entry of one row or k index: x = element offset, y = packed
// (h + bias) << 16 | (w + bias).  An index outside [lo, hi) gets h-field 0,
// which fails the box test against any partner.
__device__ inline int2 lut_entry(const AxisMap &a, int idx, int lo, int hi) {
    int2 e;
    if (idx >= lo && idx < hi) {
        int off, h, w;
        axis_decode(a, idx, off, h, w);
        e.x = off;
        e.y = ((h + HW_BIAS) << 16) | (w + HW_BIAS);
    } else {
        e.x = 0;
        e.y = HW_BIAS;
    }
    return e;
}

__device__ inline bool box_ok(int2 rp, int2 kp, int HL, int WL) {
    unsigned s = (unsigned)rp.y + (unsigned)kp.y;
    int h = (int)(s >> 16) - 2 * HW_BIAS;
    int w = (int)(s & 0xffffu) - 2 * HW_BIAS;
    return ((unsigned)h < (unsigned)HL) && ((unsigned)w < (unsigned)WL);
}

template <typename T>
union Stage {
    uint4 v[4];
    T e[64 / sizeof(T)];
};

// Fetch this thread's share of an R-row operand slab into registers.
// kl = slab start relative to the look-up window, kg = absolute slab start.
template <typename T, int R>
__device__ inline void load_stage(Stage<T> &st, const T *__restrict__ base, const OperandMap &om,
                                  const int2 *rlut, const int2 *klut, int kl, int kg, int kend,
                                  int tid) {
    constexpr int VEC = Traits<T>::VEC, BKE = Traits<T>::BKE;
    const int mode = om.mode;
    if (mode == FILL_VEC_K) {
        constexpr int NCH = (R * 4 + 255) / 256;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            int c = tid + i * 256;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (c < R * 4) {
                int row = c >> 2, kc = c & 3;
                int2 rp = rlut[row];
                int2 kp = klut[kl + kc * VEC];
                if ((rp.y >> 16) != 0 && (kp.y >> 16) != 0)
                    v = *reinterpret_cast<const uint4 *>(base + rp.x + kp.x);
            }
            st.v[i] = v;
        }
    } else if (mode == FILL_VEC_R) {
        constexpr int RV = R / VEC;  // row vectors per k
        if (tid < R) {
            int rv = tid % RV, kq = tid / RV;
            int2 rp = rlut[rv * VEC];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int2 kp = klut[kl + kq * 4 + i];
                uint4 v = make_uint4(0, 0, 0, 0);
                if ((rp.y >> 16) != 0 && (kp.y >> 16) != 0)
                    v = *reinterpret_cast<const uint4 *>(base + rp.x + kp.x);
                st.v[i] = v;
            }
        }
    } else if (mode == FILL_ELEM_R) {
        constexpr int SLOTS = 256 / R, PER = BKE / SLOTS;
        int row = tid % R, slot = tid / R;
        int2 rp = rlut[row];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            int2 kp = klut[kl + slot + j * SLOTS];
            T x = (T)0;
            if (box_ok(rp, kp, om.HL, om.WL)) x = base[rp.x + kp.x];
            st.e[j] = x;
        }
    } else {  // FILL_ELEM_K
        constexpr int RSLOTS = 256 / BKE, PER = R / RSLOTS;
        int kk = tid % BKE, rs = tid / BKE;
        int2 kp = klut[kl + kk];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            int2 rp = rlut[rs + j * RSLOTS];
            T x = (T)0;
            if (box_ok(rp, kp, om.HL, om.WL)) x = base[rp.x + kp.x];
            st.e[j] = x;
        }
    }
}

// Write the staged registers into an LDS tile (rows k-contiguous, PITCH bytes).
template <typename T, int R>
__device__ inline void store_stage(const Stage<T> &st, char *tile, int mode, int tid) {
    constexpr int VEC = Traits<T>::VEC, BKE = Traits<T>::BKE;
    if (mode == FILL_VEC_K) {
        constexpr int NCH = (R * 4 + 255) / 256;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            int c = tid + i * 256;
            if (c < R * 4) {
                int row = c >> 2, kc = c & 3;
                *reinterpret_cast<uint4 *>(tile + row * PITCH + kc * 16) = st.v[i];
            }
        }
    } else if (mode == FILL_VEC_R) {
        constexpr int RV = R / VEC;
        if (tid < R) {
            int rv = tid % RV, kq = tid / RV;
            // st.v[i] holds VEC consecutive rows at k = kq*4 + i: transpose to
            // one 4-wide k run per row.
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                alignas(16) T q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) q[i] = st.e[i * VEC + j];
                char *p = tile + (rv * VEC + j) * PITCH + kq * 4 * (int)sizeof(T);
                if (sizeof(T) == 4) {
                    *reinterpret_cast<uint4 *>(p) = *reinterpret_cast<const uint4 *>(q);
                } else {
                    *reinterpret_cast<uint2 *>(p) = *reinterpret_cast<const uint2 *>(q);
                }
            }
        }
    } else if (mode == FILL_ELEM_R) {
        constexpr int SLOTS = 256 / R, PER = BKE / SLOTS;
        int row = tid % R, slot = tid / R;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            *reinterpret_cast<T *>(tile + row * PITCH + (slot + j * SLOTS) * (int)sizeof(T)) = st.e[j];
    } else {
        constexpr int RSLOTS = 256 / BKE, PER = R / RSLOTS;
        int kk = tid % BKE, rs = tid / BKE;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            *reinterpret_cast<T *>(tile + (rs + j * RSLOTS) * PITCH + kk * (int)sizeof(T)) = st.e[j];
    }
}

template <typename T>
__device__ inline void mfma_slab(f32x16 &acc, const uint4 &a, const uint4 &b);

template <>
__device__ inline void mfma_slab<half_t>(f32x16 &acc, const uint4 &a, const uint4 &b) {
    f16x8 av = __builtin_bit_cast(f16x8, a);
    f16x8 bv = __builtin_bit_cast(f16x8, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
}

template <>
__device__ inline void mfma_slab<float>(f32x16 &acc, const uint4 &a, const uint4 &b) {
    f32x4 av = __builtin_bit_cast(f32x4, a);
    f32x4 bv = __builtin_bit_cast(f32x4, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, bv.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, bv.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, bv.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, bv.w, acc, 0, 0, 0);
}

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(256) void gemm_kernel(const GemmArgs g) {
    constexpr int BKE = Traits<T>::BKE;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    constexpr int FM = WM / 32, FN = WN / 32;
    static_assert(WAVES_M * WAVES_N == 4, "four waves per workgroup");
    static_assert(FM >= 1 && FN >= 1, "wave tile is a multiple of 32x32");

    __shared__ __attribute__((aligned(16))) char tileA[2][BM * PITCH];
    __shared__ __attribute__((aligned(16))) char tileB[2][BN * PITCH];
    __shared__ int2 rlutA[BM];
    __shared__ int2 rlutB[BN];
    __shared__ int2 klutA[KW];
    __shared__ int2 klutB[KW];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    const int tile = blockIdx.x;
    const int z = blockIdx.y;
    const int tn = tile / g.tiles_m, tm = tile % g.tiles_m;
    const int n0 = tn * BM, m0 = tm * BN;
    const int kbeg = z * g.kchunk;
    const int kend = min(g.K, kbeg + g.kchunk);

    const T *__restrict__ Ab = reinterpret_cast<const T *>(g.A);
    const T *__restrict__ Bb = reinterpret_cast<const T *>(g.B);

    for (int i = tid; i < BM; i += 256) rlutA[i] = lut_entry(g.a.row, n0 + i, 0, g.N);
    for (int i = tid; i < BN; i += 256) rlutB[i] = lut_entry(g.b.row, m0 + i, 0, g.M);

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    const int a_mode = g.a.mode, b_mode = g.b.mode;
    const int frag_off = (lane & 31) * PITCH + (lane >> 5) * 16;

    for (int kw = kbeg; kw < kend; kw += KW) {
        const int kwe = min(kw + KW, kend);
        __syncthreads();
        for (int i = tid; i < KW; i += 256) {
            klutA[i] = lut_entry(g.a.k, kw + i, kw, kwe);
            klutB[i] = lut_entry(g.b.k, kw + i, kw, kwe);
        }
        __syncthreads();
        const int nsteps = (kwe - kw + BKE - 1) / BKE;

        Stage<T> sa, sb;
        load_stage<T, BM>(sa, Ab, g.a, rlutA, klutA, 0, kw, kwe, tid);
        load_stage<T, BN>(sb, Bb, g.b, rlutB, klutB, 0, kw, kwe, tid);
        store_stage<T, BM>(sa, tileA[0], a_mode, tid);
        store_stage<T, BN>(sb, tileB[0], b_mode, tid);
        __syncthreads();

        for (int s = 0; s < nsteps; ++s) {
            const bool more = (s + 1 < nsteps);
            if (more) {
                load_stage<T, BM>(sa, Ab, g.a, rlutA, klutA, (s + 1) * BKE, kw + (s + 1) * BKE, kwe, tid);
                load_stage<T, BN>(sb, Bb, g.b, rlutB, klutB, (s + 1) * BKE, kw + (s + 1) * BKE, kwe, tid);
            }
            const char *pa = tileA[s & 1] + wm * WM * PITCH + frag_off;
            const char *pb = tileB[s & 1] + wn * WN * PITCH + frag_off;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint4 af[FM], bf[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    af[i] = *reinterpret_cast<const uint4 *>(pa + i * 32 * PITCH + h * 32);
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    bf[j] = *reinterpret_cast<const uint4 *>(pb + j * 32 * PITCH + h * 32);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) mfma_slab<T>(acc[i][j], af[i], bf[j]);
            }
            if (more) {
                store_stage<T, BM>(sa, tileA[(s + 1) & 1], a_mode, tid);
                store_stage<T, BN>(sb, tileB[(s + 1) & 1], b_mode, tid);
            }
            __syncthreads();
        }
    }

    // Epilogue.  Accumulator element v of fragment (i, j) in lane l is
    // C[row 8*(v/4) + 4*(l/32) + v%4][col l%32] of that 32x32 block.
    __syncthreads();
    int *nlut = reinterpret_cast<int *>(klutA);
    int *mlut = reinterpret_cast<int *>(klutB);
    if (g.splits == 1) {
        for (int i = tid; i < BM; i += 256) {
            int off = 0, h, w;
            if (n0 + i < g.N) axis_decode(g.c.n, n0 + i, off, h, w);
            nlut[i] = off;
        }
        for (int i = tid; i < BN; i += 256) {
            int off = 0, h, w;
            if (m0 + i < g.M) axis_decode(g.c.m, m0 + i, off, h, w);
            mlut[i] = off;
        }
        __syncthreads();
        T *__restrict__ Cb = reinterpret_cast<T *>(g.C);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int ml = wn * WN + j * 32 + (lane & 31);
                if (m0 + ml < g.M) {
                    int mo = mlut[ml];
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        int nl = wm * WM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                        if (n0 + nl < g.N) Cb[nlut[nl] + mo] = (T)acc[i][j][v];
                    }
                }
            }
    } else {
        float *__restrict__ ws = g.ws + (size_t)z * g.N * g.M;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int m = m0 + wn * WN + j * 32 + (lane & 31);
                if (m < g.M) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        int n = n0 + wm * WM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                        if (n < g.N) ws[(size_t)n * g.M + m] = acc[i][j][v];
                    }
                }
            }
    }
}

// Sum split-K partials (fixed order) and scatter through the output map: 64 outputs per
// workgroup, four split groups in parallel, four loads in flight per thread -- with few outputs
// and many splits the kernel lives on memory-level parallelism.
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ ws, T *__restrict__ C,
                                                            OutMap c, int N, int M, int splits, const T *__restrict__ bias) {
    __shared__ float part[4][64];
    const size_t total = (size_t)N * M;
    const int o = threadIdx.x & 63, sg = threadIdx.x >> 6;
    const size_t idx = (size_t)blockIdx.x * 64 + o;
    float s = 0.f;
    if (idx < total) {
        const float *src = ws + idx;
        int z = sg;
        for (; z + 3 * 4 < splits; z += 4 * 4) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[(size_t)(z + u * 4) * total];
#pragma unroll
            for (int u = 0; u < 4; ++u) s += v[u];
        }
        for (; z < splits; z += 4) s += src[(size_t)z * total];
    }
    part[sg][o] = s;
    __syncthreads();
    if (sg != 0 || idx >= total) return;
    s += part[1][o] + part[2][o] + part[3][o];
    int n = (int)(idx / M), m = (int)(idx % M);
    int on, om, h, w;
    axis_decode(c.n, n, on, h, w);
    axis_decode(c.m, m, om, h, w);
    if (bias) s += (float)bias[m];
    C[on + om] = (T)s;
}

// The bias of a product that the register-staged kernel has stored.
template <typename T>
__global__ __launch_bounds__(256) void bias_map_kernel(T *__restrict__ C, OutMap c, int N, int M, const T *__restrict__ bias) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)N * M) return;
    const int n = (int)(idx / M), m = (int)(idx % M);
    int on, om, h, w;
    axis_decode(c.n, n, on, h, w);
    axis_decode(c.m, m, om, h, w);
    C[on + om] = (T)((float)C[on + om] + (float)bias[m]);
}

// ---------------------------------------------------------------------------
// Host side: operand fill mode, tile shape and split selection, launch.
// ---------------------------------------------------------------------------
static bool axis_is_single(const AxisMap &a) { return a.d0 >= a.n; }

static bool no_coords(const AxisMap &a) {
    return a.h2 == 0 && a.h1 == 0 && a.h0 == 0 && a.hb == 0 && a.w2 == 0 && a.w1 == 0 && a.w0 == 0 &&
           a.wb == 0;
}

static bool mult(const AxisMap &a, int v, bool include_o0) {
    return a.o2 % v == 0 && a.o1 % v == 0 && a.ob % v == 0 && (!include_o0 || a.o0 % v == 0);
}

template <typename T>
static int choose_mode(const OperandMap &om, const void *base, int rows, int K) {
    constexpr int VEC = Traits<T>::VEC;
    bool plain_box = no_coords(om.row) && no_coords(om.k) && om.HL >= 1 && om.WL >= 1;
    bool aligned = (reinterpret_cast<uintptr_t>(base) % 16) == 0;
    if (plain_box && aligned) {
        // contiguous along k: a 16-byte vector must stay inside one q0 run
        if (om.k.o0 == 1 && (axis_is_single(om.k) || om.k.d0 % VEC == 0) && K % VEC == 0 &&
            mult(om.k, VEC, false) && mult(om.row, VEC, true))
            return FILL_VEC_K;
        if (om.row.o0 == 1 && (axis_is_single(om.row) || om.row.d0 % VEC == 0) && rows % VEC == 0 &&
            mult(om.row, VEC, false) && mult(om.k, VEC, true))
            return FILL_VEC_R;
    }
    // Element gather: consecutive lanes walk the axis whose unit-stride runs are longer (for an
    // implicit im2col that is the pixel axis: a row of the image against a row of the filter).
    auto run = [](const AxisMap &a) {
        int s = a.o0 < 0 ? -a.o0 : a.o0;
        int len = a.d0 < a.n ? a.d0 : a.n;
        return s == 1 ? len : 0;
    };
    int rk = run(om.k), rr = run(om.row);
    if (rk != rr) return rk > rr ? FILL_ELEM_K : FILL_ELEM_R;
    int ak = om.k.o0 < 0 ? -om.k.o0 : om.k.o0;
    int ar = om.row.o0 < 0 ? -om.row.o0 : om.row.o0;
    return ak <= ar ? FILL_ELEM_K : FILL_ELEM_R;
}

template <typename T, int BM, int BN, int WMv, int WNv>
static void launch_cfg(GemmArgs &g, hipStream_t s) {
    g.tiles_n = (g.N + BM - 1) / BM;
    g.tiles_m = (g.M + BN - 1) / BN;
    dim3 grid(g.tiles_n * g.tiles_m, g.splits);
    hipLaunchKernelGGL((gemm_kernel<T, BM, BN, WMv, WNv>), grid, dim3(256), 0, s, g);
}

// Tile shape, split selection and launch of the staged kernel.
template <typename T>
static int launch_staged(GemmArgs &g) {
    State &st = state();
    constexpr int BKE = Traits<T>::BKE;
    // Tile shape: skinny outputs get a 32-row (or 32-column) tile; otherwise the
    // largest square tile that still yields at least one workgroup per CU.
    int cfg;
    auto tiles = [&](int bm, int bn) { return (long)((g.N + bm - 1) / bm) * ((g.M + bn - 1) / bn); };
    if (g.N <= 32)
        cfg = 2;
    else if (g.M <= 32)
        cfg = 3;
    else if (tiles(128, 128) >= st.num_cu)
        cfg = 0;
    else
        cfg = 1;
    long nt = cfg == 0 ? tiles(128, 128) : cfg == 1 ? tiles(64, 64) : cfg == 2 ? tiles(32, 128) : tiles(128, 32);

    // Split k when the output alone cannot fill the machine.
    g.splits = 1;
    g.kchunk = ((g.K + BKE - 1) / BKE) * BKE;
    if (nt * 2 <= st.num_cu) {
        int min_chunk = 4 * BKE;
        int max_splits = (g.K + min_chunk - 1) / min_chunk;
        int want = (int)((st.num_cu + nt - 1) / nt);
        int sp = want < max_splits ? want : max_splits;
        if (sp > 1) {
            int chunk = (g.K + sp - 1) / sp;
            chunk = ((chunk + BKE - 1) / BKE) * BKE;
            sp = (g.K + chunk - 1) / chunk;
            if (sp > 1) {
                g.splits = sp;
                g.kchunk = chunk;
            }
        }
    }
    if (g.splits > 1) {
        g.ws = workspace((size_t)g.splits * g.N * g.M * sizeof(float));
        if (!g.ws) return 2;
    }
    switch (cfg) {
        case 0: launch_cfg<T, 128, 128, 2, 2>(g, st.stream); break;
        case 1: launch_cfg<T, 64, 64, 2, 2>(g, st.stream); break;
        case 2: launch_cfg<T, 32, 128, 1, 4>(g, st.stream); break;
        default: launch_cfg<T, 128, 32, 4, 1>(g, st.stream); break;
    }
    return hip_ok(hipGetLastError(), "gemm launch") ? 0 : 2;
}

// The product as the kernel for any size and alignment takes it: both operands matrices that are contiguous along k or
// along their rows, k a single axis or runs of one (sample, pixel), the rows of one operand likewise.  -1: not such a
// product.
template <typename T>
static int gemm_ragged(const GemmArgs &gin) {
    constexpr long long ES = (long long)sizeof(T);
    GemmArgs g = gin;
    bool swapped = false;
    auto two = [](const AxisMap &a) { return !axis_is_single(a); };
    // the operand whose rows have two digits, and the one along which the output is contiguous, go second
    if (two(g.a.row) || (!two(g.b.row) && g.c.m.o0 != 1 && g.c.n.o0 == 1)) {
        GemmArgs t = g;
        t.A = g.B; t.B = g.A; t.a = g.b; t.b = g.a; t.N = g.M; t.M = g.N; t.c.n = g.c.m; t.c.m = g.c.n;
        g = t;
        swapped = true;
    }
    auto simple = [](const AxisMap &a) { return axis_is_single(a) || (a.d1 >= (1 << 30) && a.n % a.d0 == 0); };
    if (!simple(g.a.k) || !simple(g.b.k) || !axis_is_single(g.a.row) || !simple(g.b.row) || !simple(g.c.m) || !axis_is_single(g.c.n)) return -1;
    if (!no_coords(g.a.row) || !no_coords(g.a.k) || !no_coords(g.b.row) || !no_coords(g.b.k) || g.taps > 1) return -1;
    if (two(g.a.k) != two(g.b.k) || (two(g.a.k) && g.a.k.d0 != g.b.k.d0) || two(g.b.row) != two(g.c.m) ||
        (two(g.b.row) && g.b.row.d0 != g.c.m.d0) || g.c.n.ob || g.c.m.ob)
        return -1;
    RagArgs r = {};
    RagProd &p = r.p[0];
    r.count = 1;
    p.N = g.N;
    p.M = g.M;
    p.K = two(g.a.k) ? g.a.k.d0 : g.K;
    p.runs = g.K / p.K;
    p.m_in = two(g.b.row) ? g.b.row.d0 : g.M;
    p.outer = g.M / p.m_in;
    auto operand = [&](const OperandMap &o, const void *base, int rows, RagOp &q) {
        const AxisMap &row = o.row, &k = o.k;
        const int in = axis_is_single(row) ? rows : row.d0;
        if (row.ob < 0 || k.ob < 0 || row.o0 <= 0 || k.o0 <= 0 || row.o1 < 0 || k.o1 < 0) return -1;
        if (k.o0 != 1 && row.o0 != 1) return -1;
        if ((long long)row.o0 * ES >= (1ll << 24) || (long long)k.o0 * ES >= (1ll << 24)) return -1;  // (128 rows in 32 bits)
        q.p = reinterpret_cast<const char *>(base) + (row.ob + (long long)k.ob) * ES;
        q.rows = in;
        q.row_b = (unsigned)(row.o0 * ES);
        q.k_b = (unsigned)(k.o0 * ES);
        q.run_b = p.runs > 1 ? (long long)k.o1 * ES : 0;
        q.outer_b = in < rows ? (long long)row.o1 * ES : 0;
        // (a piece must fit into the contiguous run it is read from)
        constexpr int VEC = 16 / (int)sizeof(T);
        const bool kc = k.o0 == 1 && p.K >= VEC, rc = row.o0 == 1 && in >= VEC;
        return kc && (!rc || p.K >= in) ? (int)RAG_KC : rc ? (int)RAG_RC : -1;
    };
    const int am = operand(g.a, g.A, g.N, p.a), bm = operand(g.b, g.B, g.M, p.b);
    if (am < 0 || bm < 0 || (p.outer > 1 && bm != RAG_RC)) return -1;
    p.bias = g.bias;
    p.bias_n = swapped;
    p.C = g.C;
    p.cn = rag_axis(g.N, g.c.n.o0);
    p.cm = two(g.c.m) ? rag_axis2(g.c.m.d0, g.c.m.o0, g.c.m.o1) : rag_axis(g.M, g.c.m.o0);
    return ragged<T>(r, am, bm, am, bm);
}

template <typename T>
int gemm(const GemmArgs &gin) {
    if (!ensure_init()) return 2;
    GemmArgs g = gin;
    if (g.N <= 0 || g.M <= 0 || g.K <= 0) return 0;
    State &st = state();

    g.a.mode = choose_mode<T>(g.a, g.A, g.N, g.K);
    g.b.mode = choose_mode<T>(g.b, g.B, g.M, g.K);

    int rc = -1;
    if (st.gemm_path != 1) {
        // whole slabs of aligned rows: the look-up-free kernel; other matrices: the one for any size and alignment;
        // index maps with coordinates: the gathering kernel
        constexpr int SK = 128 / (int)sizeof(T);
        const bool lean_runs = g.a.mode == FILL_VEC_K && g.b.mode == FILL_VEC_K && !axis_is_single(g.a.k) && g.a.k.d0 == g.b.k.d0 &&
                               g.a.k.d0 % SK == 0;
        if (!lean_runs && !(plain_operand<T>(g.a, SK, g.K) && plain_operand<T>(g.b, SK, g.K))) {
            rc = gemm_ragged<T>(g);
            if (rc >= 0) return rc;
        }
        rc = gemm_async<T>(g);
    }
    if (rc > 0) return rc;
    if (rc < 0) {
        rc = launch_staged<T>(g);
        if (rc) return rc;
        if (g.bias && g.splits == 1) {
            hipLaunchKernelGGL((bias_map_kernel<T>), dim3((unsigned)(((size_t)g.N * g.M + 255) / 256)), dim3(256), 0, st.stream,
                               reinterpret_cast<T *>(g.C), g.c, g.N, g.M, reinterpret_cast<const T *>(g.bias));
            if (!hip_ok(hipGetLastError(), "bias add launch")) return 2;
        }
    }
    if (g.splits > 1) {
        size_t total = (size_t)g.N * g.M;
        hipLaunchKernelGGL((splitk_reduce_kernel<T>), dim3((unsigned)((total + 63) / 64)), dim3(256), 0,
                           st.stream, g.ws, reinterpret_cast<T *>(g.C), g.c, g.N, g.M, g.splits, reinterpret_cast<const T *>(g.bias));
        if (!hip_ok(hipGetLastError(), "split-k reduce launch")) return 2;
    }
    return 0;
}

template <typename T>
int gemm_pair_lean(const GemmArgs &g0in, const GemmArgs &g1in) {
    if (!ensure_init()) return 2;
    GemmArgs g0 = g0in, g1 = g1in;
    if (state().gemm_path == 0 && g0.N > 0 && g0.M > 0 && g0.K > 0 && g1.N > 0 && g1.M > 0 && g1.K > 0) {
        g0.a.mode = choose_mode<T>(g0.a, g0.A, g0.N, g0.K);
        g0.b.mode = choose_mode<T>(g0.b, g0.B, g0.M, g0.K);
        g1.a.mode = choose_mode<T>(g1.a, g1.A, g1.N, g1.K);
        g1.b.mode = choose_mode<T>(g1.b, g1.B, g1.M, g1.K);
        int rc = gemm_async_pair<T>(g0, g1);
        if (rc >= 0) return rc;
    }
    return -1;
}

template <typename T>
int gemm_pair(const GemmArgs &g0in, const GemmArgs &g1in) {
    int rc = gemm_pair_lean<T>(g0in, g1in);
    if (rc >= 0) return rc;
    rc = gemm<T>(g0in);
    return rc ? rc : gemm<T>(g1in);
}
template int gemm_pair_lean<float>(const GemmArgs &, const GemmArgs &);
template int gemm_pair_lean<half_t>(const GemmArgs &, const GemmArgs &);

// dW[o][i] = sum_b dY[b][o] X[b][i] and dX[b][i] = sum_o dY[b][o] W[o][i] and
// the bias gradient db[o] = sum_b dY[b][o] (null: none) as one launch of the kernel for any size and alignment; -1 when a
// row is shorter than its 16-byte pieces.
template <typename T>
int linear_bw_ragged(const T *X, const T *W, const T *dY, T *dW, T *dX, T *db, int ns, int in, int out) {
    constexpr int VEC = 16 / (int)sizeof(T), ES = (int)sizeof(T);
    if (in < VEC || out < VEC || in >= (1 << 22) || out >= (1 << 22)) return -1;
    auto matrix = [](const T *p, int rows, int row_stride, int k_stride) {
        RagOp q = {};
        q.p = reinterpret_cast<const char *>(p);
        q.rows = rows;
        q.row_b = (unsigned)row_stride * ES;
        q.k_b = (unsigned)k_stride * ES;
        return q;
    };
    RagArgs r = {};
    r.count = 2;
    RagProd &w = r.p[0], &x = r.p[1];
    w.a = matrix(dY, out, 1, out);
    w.b = matrix(X, in, 1, in);
    w.C = dW;
    w.N = out;
    w.M = w.m_in = in;
    w.K = ns;
    w.row_sum = db;
    w.cn = rag_axis(out, in);
    w.cm = rag_axis(in, 1);
    x.a = matrix(dY, ns, out, 1);
    x.b = matrix(W, in, 1, in);
    x.C = dX;
    x.N = ns;
    x.M = x.m_in = in;
    x.K = out;
    x.cn = rag_axis(ns, in);
    x.cm = rag_axis(in, 1);
    w.runs = x.runs = w.outer = x.outer = 1;
    return ragged<T>(r, RAG_RC, RAG_RC, RAG_KC, RAG_RC);
}
template int linear_bw_ragged<float>(const float *, const float *, const float *, float *, float *, float *, int, int, int);
template int linear_bw_ragged<half_t>(const half_t *, const half_t *, const half_t *, half_t *, half_t *, half_t *, int, int, int);

template int gemm_pair<float>(const GemmArgs &, const GemmArgs &);
template int gemm_pair<half_t>(const GemmArgs &, const GemmArgs &);
template int gemm<float>(const GemmArgs &);
template int gemm<half_t>(const GemmArgs &);

// ---------------------------------------------------------------------------
// Products with a unit dimension (Linear at batch 1): bound by the launch below about 1 MB (2.5 us of host time each),
// by memory above.  All of them read and write 16-byte pieces at any element alignment; the last piece of a row is the
// one that ends with it (columns it shares with the piece before are worked out twice, with the same result), rows
// shorter than a piece go element by element (V = 1).
// ---------------------------------------------------------------------------
constexpr int GV_NT = 512;

template <typename T, int V>
struct GvPiece {
    T e[V];
};
template <typename T, int V>
__device__ inline GvPiece<T, V> gv_load(const T *p) {
    GvPiece<T, V> v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}

// y[r] = sum_k Mx[r*K + k] * x[k] (+ bias[r]); one wave per row.
template <typename T, int V>
__global__ __launch_bounds__(256) void gemv_rowdot_kernel(const T *__restrict__ Mx, const T *__restrict__ x, T *__restrict__ y,
                                                          const T *__restrict__ bias, int R, int K) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= R) return;
    const T *p = Mx + (size_t)row * K;
    float s = 0.f;
    const int whole = K / V * V;
    for (int k = lane * V; k < whole; k += 64 * V) {
        const GvPiece<T, V> a = gv_load<T, V>(p + k), b = gv_load<T, V>(x + k);
#pragma unroll
        for (int i = 0; i < V; ++i) s += (float)a.e[i] * (float)b.e[i];
    }
    if (whole + lane < K) s += (float)p[whole + lane] * (float)x[whole + lane];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if (lane == 0) y[row] = (T)(bias ? s + (float)bias[row] : s);
}

// How the rows of a column sum are shared out: `cols` workgroups side by side, each share `chunk` rows.
struct GvShares {
    int cols, shares, chunk;
    float *part;  // [share][sample][M]; one share: the kernel writes the result
};

// Workgroup `block` sums share block / cols of eight pieces of columns (a 128-byte line: four, of which two workgroups
// on different XCDs share a line, take up to twice as long from 8 MB on) of y[m] = sum_k x[k] * Mx[k*M + m]: thread (kl, cv)
// takes rows kl, kl + 64, ... of piece cv with four loads in flight, the rows meet in LDS (first eight, then the rest).
constexpr int GV_CV = 8, GV_ROWS = GV_NT / GV_CV, GV_U = 4;
template <typename T, int V>
__device__ inline void gemv_coldot_block(const T *__restrict__ x, const T *__restrict__ Mx, T *__restrict__ y, int K, int M,
                                         int block, const GvShares &sh, float *red) {
    constexpr int CV = GV_CV, KL = GV_ROWS, U = GV_U, NT = GV_NT;
    const int share = block / sh.cols;
    block -= share * sh.cols;
    const unsigned k0 = (unsigned)share * (unsigned)sh.chunk, k1 = min((unsigned)K, k0 + (unsigned)sh.chunk);
    const int cv = threadIdx.x % CV, kl = threadIdx.x / CV;
    const int want = (block * CV + cv) * V, col = want + V <= M ? want : M - V;
    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
    if (want < M) {
        // (addresses by additions of a uniform step: a 64-bit product per load takes a fifth of the time of short columns)
        const size_t step = (size_t)KL * M;
        unsigned k = k0 + kl;
        const T *q = Mx + (size_t)k * M + col, *xq = x + k;
        for (; k + (U - 1) * KL < k1; k += U * KL, q += U * step, xq += U * KL) {
            GvPiece<T, V> v[U];
            T xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v[u] = gv_load<T, V>(q + u * step);
                xv[u] = xq[u * KL];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < V; ++i) acc[i] += (float)xv[u] * (float)v[u].e[i];
        }
        if (k < k1) {  // (rows beyond the end: the first one, replaced by zeros; a branch around them would take each load into it)
            GvPiece<T, V> v[U - 1];
            T xv[U - 1];
            bool in[U - 1];
#pragma unroll
            for (int u = 0; u < U - 1; ++u) {
                in[u] = k + u * KL < k1;
                v[u] = gv_load<T, V>(q + (in[u] ? u * step : 0));
                xv[u] = xq[in[u] ? u * KL : 0];
            }
#pragma unroll
            for (int u = 0; u < U - 1; ++u) {
                const float f = in[u] ? (float)xv[u] : 0.f;
#pragma unroll
                for (int i = 0; i < V; ++i) acc[i] += f * (in[u] ? (float)v[u].e[i] : 0.f);
            }
        }
    }
    // lanes of a wave that share a piece are CV apart
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
        for (int o = 32; o >= CV; o >>= 1) acc[i] += __shfl_xor(acc[i], o, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < CV) {
#pragma unroll
        for (int i = 0; i < V; ++i) red[wave * (CV * V) + lane * V + i] = acc[i];
    }
    __syncthreads();
    if ((int)threadIdx.x < CV * V) {
        const int c = threadIdx.x / V, first = (block * CV + c) * V, at = (first + V <= M ? first : M - V) + threadIdx.x % V;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) s += red[w * (CV * V) + threadIdx.x];
        if (first < M) {
            if (sh.shares > 1) sh.part[(size_t)share * M + at] = s;
            else y[at] = (T)s;
        }
    }
}

template <typename T, int V>
__global__ __launch_bounds__(GV_NT) void gemv_coldot_kernel(const T *__restrict__ x, const T *__restrict__ Mx, T *__restrict__ y,
                                                            int K, int M, const GvShares sh) {
    __shared__ float red[GV_NT / 64 * GV_CV * V];
    gemv_coldot_block<T, V>(x, Mx, y, K, M, blockIdx.x, sh, red);
}

// C[n*M + m] = a[n] * b[m]: unit `i` is a piece of columns of four consecutive rows; the first piece of a row also copies
// a[n] to `copy` where that is wanted (the bias gradient of one sample).
template <typename T, int V>
__device__ inline void outer_unit(const T *__restrict__ a, const T *__restrict__ b, T *__restrict__ C, T *__restrict__ copy,
                                  int N, int M, RagDiv per_row, unsigned i) {
    const unsigned q = per_row.m ? __umulhi(i, per_row.m) >> per_row.s : i;
    const int n0 = (int)q * 4, want = (int)(i - q * per_row.d) * V;
    if (n0 >= N) return;
    const int m = want + V <= M ? want : M - V;
    const GvPiece<T, V> bv = gv_load<T, V>(b + m);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (n0 + r >= N) break;
        const T an = a[n0 + r];
        const float av = (float)an;
        GvPiece<T, V> out;
#pragma unroll
        for (int e = 0; e < V; ++e) out.e[e] = (T)(av * (float)bv.e[e]);
        __builtin_memcpy(C + (size_t)(n0 + r) * M + m, &out, sizeof(out));
        if (copy && want == 0) copy[n0 + r] = an;
    }
}

template <typename T, int V>
__global__ __launch_bounds__(GV_NT) void outer_kernel(const T *__restrict__ a, const T *__restrict__ b, T *__restrict__ C, int N,
                                                      int M, RagDiv per_row) {
    outer_unit<T, V>(a, b, C, nullptr, N, M, per_row, blockIdx.x * GV_NT + threadIdx.x);
}

// Both gradients of a dense layer on one sample in one launch (1024 x 1024 in fp32: 5.9 us as two launches, bound by the
// host; 3.3 as one): the first workgroups sum columns for dX, the rest write dW (and db = dY).
template <typename T, int V>
__global__ __launch_bounds__(GV_NT) void linear_one_bw_kernel(const T *__restrict__ x, const T *__restrict__ W,
                                                              const T *__restrict__ dy, T *__restrict__ dW, T *__restrict__ dx,
                                                              T *__restrict__ db, int in, int out, RagDiv per_row,
                                                              const GvShares sh) {
    __shared__ float red[GV_NT / 64 * GV_CV * V];
    const int sums = sh.cols * sh.shares;
    if ((int)blockIdx.x < sums)
        gemv_coldot_block<T, V>(dy, W, dx, out, in, blockIdx.x, sh, red);
    else
        outer_unit<T, V>(dy, x, dW, db, out, in, per_row, (blockIdx.x - sums) * GV_NT + threadIdx.x);
}

// Few columns leave CUs without a workgroup, and a workgroup has a trip to memory for every 256 of its rows.  Columns of 4096
// rows and more are shared out over two workgroups a CU, 512 rows and more each, at most 32 shares, where that is two
// shares at least; adding them is a launch (2.3 us).  In us, one share against these, fp32: 64 columns of 2048 rows 4.0, 6.1
// (not taken), of 4096 6.8, 6.1, of 16384 25.3, 6.4; 1024 columns of 2048 rows 5.8, 6.6 (not taken), of 4096 9.9, 6.7; 4096
// of 4096 18.8, 15.7; 6144 of 4096 21.5, 21.9 (not taken).
// With several samples the sums themselves take a workgroup 1.7 us for every 512 rows: shares from FEW_SHARED rows on (5
// samples, 1152 -> 3328 in fp16 22.5 us with one share, 12.3 with six).
constexpr int FEW_SHARED = 1536;
template <typename T, int V>
static GvShares gv_shares(int K, int M, int ns = 1) {
    GvShares sh = {(int)(((long long)M + GV_CV * V - 1) / (GV_CV * V)), 1, K, nullptr};
    const int cu = state().num_cu, z = std::min({2 * cu / sh.cols, K / 512, 32});
    if (K < (ns > 1 ? FEW_SHARED : 4096) || sh.cols > cu / 2 || z < 2) return sh;
    const int chunk = (K + z - 1) / z, shares = (K + chunk - 1) / chunk;
    // (a stream that is being captured, or a full device, cannot get a workspace: one share then)
    if (float *part = workspace_if((size_t)shares * ns * M * sizeof(float))) sh = {sh.cols, shares, chunk, part};
    return sh;
}

static unsigned outer_blocks(int N, int M, int V) {
    return (unsigned)(((size_t)((N + 3) / 4) * ((M + V - 1) / V) + GV_NT - 1) / GV_NT);
}

// (a launch takes the rows whose units are 31-bit numbers: all of them below 2^35 outputs of 4 bytes)
template <typename T, int V>
static int outer(const T *a, const T *b, T *C, int N, int M) {
    const RagDiv per_row = rag_div((M + V - 1) / V);
    const long long most = ((1ll << 31) - GV_NT) / per_row.d * 4;
    for (long long n = 0; n < N; n += most) {
        const int rows = (int)(N - n < most ? N - n : most);
        hipLaunchKernelGGL((outer_kernel<T, V>), dim3(outer_blocks(rows, M, V)), dim3(GV_NT), 0, state().stream, a + n, b,
                           C + (size_t)n * M, rows, M, per_row);
    }
    return hip_ok(hipGetLastError(), "outer launch") ? 0 : 2;
}

template <typename T, int V>
static int linear_one_bw_v(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int in, int out) {
    const GvShares sh = gv_shares<T, V>(out, in);
    hipLaunchKernelGGL((linear_one_bw_kernel<T, V>), dim3(sh.cols * sh.shares + outer_blocks(out, in, V)), dim3(GV_NT), 0,
                       state().stream, x, W, dy, dW, dx, db, in, out, rag_div((in + V - 1) / V), sh);
    if (sh.shares > 1) launch_share_sum<T>(sh.part, dx, in, sh.shares, state().stream);
    return hip_ok(hipGetLastError(), "linear backward launch") ? 0 : 2;
}
template <typename T>
int linear_one_bw(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int in, int out) {
    constexpr int VEC = Traits<T>::VEC;
    return in >= VEC ? linear_one_bw_v<T, VEC>(x, W, dy, dW, dx, db, in, out) : linear_one_bw_v<T, 1>(x, W, dy, dW, dx, db, in, out);
}
template int linear_one_bw<float>(const float *, const float *, const float *, float *, float *, float *, int, int);
template int linear_one_bw<half_t>(const half_t *, const half_t *, const half_t *, half_t *, half_t *, half_t *, int, int);

// ---- dense layers on a few samples ----------------------------------------------------------------------------------
// The weights are read, their gradient is written once for all samples; 32 x 32 MFMA tiles would be three quarters padding or
// more, and a contraction that few tiles share needs partial sums and a second launch.  Sums in fp32 as with one sample.  Bound
// by a launch and two or three trips to memory up to some MB (3.5 us forward, 4.2 backward), by memory above (3595 -> 3776, 3
// samples, fp16, backward 24 us, 54 MB; before 30).

// y[b][r] = sum_k W[r][k] * x[b][k] (+ bias[r]): WPR waves a row, a piece of the row and of each sample a lane.
template <typename T, int V, int NS, int WPR>
__global__ __launch_bounds__(256) void linear_few_fw_kernel(const T *__restrict__ W, const T *__restrict__ x, T *__restrict__ y,
                                                            const T *__restrict__ bias, int ns, int in, int out) {
    constexpr int U = NS <= 4 ? 4 : 2, STEP = WPR * 64 * V;
    __shared__ float red[4][NS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * (4 / WPR) + wave / WPR, part = wave % WPR;
    float s[NS];
#pragma unroll
    for (int b = 0; b < NS; ++b) s[b] = 0.f;
    if (row < out) {
        const T *p = W + (size_t)row * in, *xb[NS];
#pragma unroll
        for (int b = 0; b < NS; ++b) xb[b] = x + (size_t)min(b, ns - 1) * in;
        const int whole = in / V * V;
        int k = (part * 64 + lane) * V;
        for (; k + (U - 1) * STEP < whole; k += U * STEP) {
            GvPiece<T, V> w[U], v[U][NS];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                w[u] = gv_load<T, V>(p + k + u * STEP);
#pragma unroll
                for (int b = 0; b < NS; ++b) v[u][b] = gv_load<T, V>(xb[b] + k + u * STEP);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int b = 0; b < NS; ++b)
#pragma unroll
                    for (int i = 0; i < V; ++i) s[b] += (float)w[u].e[i] * (float)v[u][b].e[i];
        }
        if (k < whole) {  // (pieces beyond the end: the first one, replaced by zeros)
            GvPiece<T, V> w[U - 1], v[U - 1][NS];
            bool ok[U - 1];
#pragma unroll
            for (int u = 0; u < U - 1; ++u) {
                ok[u] = k + u * STEP < whole;
                const int at = ok[u] ? k + u * STEP : k;
                w[u] = gv_load<T, V>(p + at);
#pragma unroll
                for (int b = 0; b < NS; ++b) v[u][b] = gv_load<T, V>(xb[b] + at);
            }
#pragma unroll
            for (int u = 0; u < U - 1; ++u)
#pragma unroll
                for (int b = 0; b < NS; ++b)
#pragma unroll
                    for (int i = 0; i < V; ++i) s[b] += (ok[u] ? (float)w[u].e[i] : 0.f) * (ok[u] ? (float)v[u][b].e[i] : 0.f);
        }
        if (part == 0 && whole + lane < in) {
#pragma unroll
            for (int b = 0; b < NS; ++b) s[b] += (float)p[whole + lane] * (float)xb[b][whole + lane];
        }
    }
#pragma unroll
    for (int b = 0; b < NS; ++b)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s[b] += __shfl_xor(s[b], o, 64);
    float v = s[0];  // lane b: of sample b
#pragma unroll
    for (int b = 1; b < NS; ++b) v = lane == b ? s[b] : v;
    if constexpr (WPR > 1) {
        if (lane < NS) red[wave][lane] = v;
        __syncthreads();
        if (part == 0 && lane < NS) {
            v = red[wave][lane];
#pragma unroll
            for (int w = 1; w < WPR; ++w) v += red[wave + w][lane];
        }
    }
    if (part == 0 && lane < ns && row < out) y[(size_t)lane * out + row] = (T)(bias ? v + (float)bias[row] : v);
}

// dx[b][m] = sum_k dy[b][k] * W[k][m], as gemv_coldot_block for one sample: eight rows a thread and trip, the dy's of the 512 rows
// of a trip in LDS, those of a row side by side.
template <typename T, int V, int NS>
struct FewSums {
    static constexpr int U = 8, ROWS = U * GV_ROWS, WAVES = GV_NT / 64, RED = NS * WAVES * GV_CV * V, DY = ROWS * NS;
    static constexpr int FLOATS = RED > DY ? RED : DY;
    static_assert(ROWS == GV_NT, "a thread fetches the dy's of a row");
};
template <typename T, int V, int NS>
__device__ inline void linear_few_sums(const T *__restrict__ dy, const T *__restrict__ W, T *__restrict__ dx, int ns, int K, int M, int block,
                                       const GvShares &sh, float *lds) {
    typedef FewSums<T, V, NS> S;
    constexpr int CV = GV_CV, KL = GV_ROWS, U = S::U, NT = GV_NT;
    const int share = block / sh.cols;
    block -= share * sh.cols;
    const int k0 = share * sh.chunk, k1 = min(K, k0 + sh.chunk);
    const int tid = threadIdx.x, cv = tid % CV, kl = tid / CV;
    const int want = (block * CV + cv) * V, col = min(want, M - V);
    float acc[NS][V];
#pragma unroll
    for (int b = 0; b < NS; ++b)
#pragma unroll
        for (int i = 0; i < V; ++i) acc[b][i] = 0.f;
    for (int c = k0; c < k1; c += S::ROWS) {
        const bool whole = c + S::ROWS <= k1;  // (rows beyond the end: the last one, replaced by zeros)
        GvPiece<T, V> v[U];
        T d[NS];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = gv_load<T, V>(W + (size_t)min(c + kl + u * KL, k1 - 1) * M + col);
#pragma unroll
        for (int b = 0; b < NS; ++b) d[b] = dy[(size_t)min(b, ns - 1) * K + min(c + tid, k1 - 1)];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NS; ++b) lds[tid * NS + b] = c + tid < k1 ? (float)d[b] : 0.f;
        __syncthreads();
        if (!whole) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < V; ++i) v[u].e[i] = c + kl + u * KL < k1 ? v[u].e[i] : (T)0.f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c + u * KL >= k1) break;
#pragma unroll
            for (int b = 0; b < NS; ++b) {
                const float f = lds[(kl + u * KL) * NS + b];
#pragma unroll
                for (int i = 0; i < V; ++i) acc[b][i] += f * (float)v[u].e[i];
            }
        }
    }
    // Lanes of a wave that share a piece are CV apart.  Two values a time, half of the lanes adds up the one, half the other:
    // a quarter of the values a lane in the end (with three shuffles a value the sums alone took 5 us, 64 values a lane).
    constexpr int N = NS * V, Q = N / 4;
    static_assert(N % 4 == 0 && CV == 8, "quarters");
    const int lane = tid & 63, wave = tid >> 6;
    float two[N / 2], one[Q];
    auto value = [&](int n) { return __float_as_uint(acc[n / V][n % V]); };
#pragma unroll
    for (int n = 0; n < N / 2; ++n) {
        const auto p = __builtin_amdgcn_permlane32_swap(value(n), value(n + N / 2), false, false);
        two[n] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
#pragma unroll
    for (int n = 0; n < Q; ++n) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(two[n]), __float_as_uint(two[n + Q]), false, false);
        one[n] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        one[n] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(one[n]), 0x128, 0xf, 0xf, false));  // lane ^ 8
    }
    __syncthreads();
    if (!(lane & 8)) {
        const int first = (lane >> 5) * (N / 2) + ((lane >> 4) & 1) * Q;
#pragma unroll
        for (int n = 0; n < Q; ++n) {
            const int b = (first + n) / V, i = (first + n) % V;
            lds[(b * S::WAVES + wave) * (CV * V) + (lane & 7) * V + i] = one[n];
        }
    }
    __syncthreads();
    for (int t = tid; t < NS * CV * V; t += NT) {
        const int b = t / (CV * V), r = t % (CV * V), first = (block * CV + r / V) * V, at = min(first, M - V) + r % V;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < S::WAVES; ++w) s += lds[(b * S::WAVES + w) * (CV * V) + r];
        if (first < M && b < ns) {
            if (sh.shares > 1) sh.part[((size_t)share * ns + b) * M + at] = s;
            else dx[(size_t)b * M + at] = (T)s;
        }
    }
}

// dW[n][m] = sum_b dy[b][n] * x[b][m]: a wave takes 64 pieces of columns of FEW_ROWS rows; lane (b, row) fetches a dy, which are
// the same for all lanes.  db[n] = sum_b dy[b][n] where it is wanted (plain fp32 sums lay up to 1.45 times as far from 64 bits as those
// of the other routes).
constexpr int FEW_ROWS = 8;
template <typename T, int V, int NS>
__device__ inline void linear_few_outer(const T *__restrict__ dy, const T *__restrict__ x, T *__restrict__ dW, T *__restrict__ db, int ns,
                                        int out, int in, RagDiv per_row, unsigned unit) {
    const unsigned q = rag_quot(unit, per_row);  // units of 64 pieces
    const int n0 = (int)q * FEW_ROWS, lane = threadIdx.x & 63, want = ((int)(unit - q * per_row.d) * 64 + lane) * V;
    if (n0 >= out) return;
    const int m = min(want, in - V);
    const float mine = (float)dy[(size_t)min(lane / FEW_ROWS, ns - 1) * out + min(n0 + lane % FEW_ROWS, out - 1)];
    GvPiece<T, V> xv[NS];
#pragma unroll
    for (int b = 0; b < NS; ++b) xv[b] = gv_load<T, V>(x + (size_t)min(b, ns - 1) * in + m);
#pragma unroll
    for (int r = 0; r < FEW_ROWS; ++r) {
        float s[V];
#pragma unroll
        for (int e = 0; e < V; ++e) s[e] = 0.f;
#pragma unroll
        for (int b = 0; b < NS; ++b)
            if (b < ns) {
                const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), b * FEW_ROWS + r));
#pragma unroll
                for (int e = 0; e < V; ++e) s[e] += d * (float)xv[b].e[e];
            }
        if (n0 + r < out && want < in) {
            GvPiece<T, V> o;
#pragma unroll
            for (int e = 0; e < V; ++e) o.e[e] = (T)s[e];
            __builtin_memcpy(dW + (size_t)(n0 + r) * in + m, &o, sizeof(o));
        }
    }
    if (db && want == lane * V) {  // the first unit of its rows
        LongSum<T> sum;
        sum.clear();
#pragma unroll
        for (int b = 0; b < NS; ++b) {
            const float d = __shfl(mine, b * FEW_ROWS + lane % FEW_ROWS, 64);
            if (b < ns) sum.add(d);
        }
        if (lane < FEW_ROWS && n0 + lane < out) db[n0 + lane] = (T)sum.value();
    }
}

// Both gradients in one launch: the first workgroups sum columns for dX, the rest write dW and db.
template <typename T, int V, int NS>
__global__ __launch_bounds__(GV_NT) void linear_few_bw_kernel(const T *__restrict__ x, const T *__restrict__ W, const T *__restrict__ dy,
                                                              T *__restrict__ dW, T *__restrict__ dx, T *__restrict__ db, int ns, int in,
                                                              int out, RagDiv per_row, const GvShares sh) {
    __shared__ __attribute__((aligned(16))) float lds[FewSums<T, V, NS>::FLOATS];
    const int sums = sh.cols * sh.shares;
    if ((int)blockIdx.x < sums)
        linear_few_sums<T, V, NS>(dy, W, dx, ns, out, in, blockIdx.x, sh, lds);
    else
        linear_few_outer<T, V, NS>(dy, x, dW, db, ns, out, in, per_row,
                                   (blockIdx.x - sums) * (GV_NT / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}

template <typename T, int V, int NS>
static int linear_few_bw_run(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int ns, int in, int out) {
    state().last_gemm_form = 3;
    const GvShares sh = gv_shares<T, V>(out, in, ns);
    const int per_row = (in + 64 * V - 1) / (64 * V);
    const long long units = (long long)((out + FEW_ROWS - 1) / FEW_ROWS) * per_row;
    hipLaunchKernelGGL((linear_few_bw_kernel<T, V, NS>), dim3((unsigned)(sh.cols * sh.shares + (units + GV_NT / 64 - 1) / (GV_NT / 64))),
                       dim3(GV_NT), 0, state().stream, x, W, dy, dW, dx, db, ns, in, out, rag_div(per_row), sh);
    if (sh.shares > 1) launch_share_sum<T>(sh.part, dx, ns * in, sh.shares, state().stream);
    return hip_ok(hipGetLastError(), "linear backward launch") ? 0 : 2;
}
template <typename T, int V>
static int linear_few_bw_v(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int ns, int in, int out) {
    return ns <= 2 && V > 1 ? linear_few_bw_run<T, V, (V > 1 ? 2 : 4)>(x, W, dy, dW, dx, db, ns, in, out)
         : ns <= 4 ? linear_few_bw_run<T, V, 4>(x, W, dy, dW, dx, db, ns, in, out)
                   : linear_few_bw_run<T, V, 8>(x, W, dy, dW, dx, db, ns, in, out);
}
template <typename T>
int linear_few_bw(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int ns, int in, int out) {
    constexpr int VEC = Traits<T>::VEC;
    return in >= VEC ? linear_few_bw_v<T, VEC>(x, W, dy, dW, dx, db, ns, in, out) : linear_few_bw_v<T, 1>(x, W, dy, dW, dx, db, ns, in, out);
}
template int linear_few_bw<float>(const float *, const float *, const float *, float *, float *, float *, int, int, int);
template int linear_few_bw<half_t>(const half_t *, const half_t *, const half_t *, half_t *, half_t *, half_t *, int, int, int);

template <typename T, int NS>
static int linear_few_fw_run(const T *x, const T *W, T *y, const T *bias, int ns, int in, int out) {
    constexpr int V = Traits<T>::VEC;
    hipStream_t s = state().stream;
    state().last_gemm_form = 3;
    // (rows that would not fill the chip with a wave each, and are long: four waves a row)
    if (out < 8 * state().num_cu && in > 256 * V)
        hipLaunchKernelGGL((linear_few_fw_kernel<T, V, NS, 4>), dim3(out), dim3(256), 0, s, W, x, y, bias, ns, in, out);
    else
        hipLaunchKernelGGL((linear_few_fw_kernel<T, V, NS, 1>), dim3((out + 3) / 4), dim3(256), 0, s, W, x, y, bias, ns, in, out);
    return hip_ok(hipGetLastError(), "linear forward launch") ? 0 : 2;
}
template <typename T>
int linear_few_fw(const T *x, const T *W, T *y, const T *bias, int ns, int in, int out) {
    return ns <= 2 ? linear_few_fw_run<T, 2>(x, W, y, bias, ns, in, out) : ns <= 4 ? linear_few_fw_run<T, 4>(x, W, y, bias, ns, in, out)
         : ns <= 8 ? linear_few_fw_run<T, 8>(x, W, y, bias, ns, in, out)
                   : linear_few_fw_run<T, 16>(x, W, y, bias, ns, in, out);
}
template int linear_few_fw<float>(const float *, const float *, float *, const float *, int, int, int);
template int linear_few_fw<half_t>(const half_t *, const half_t *, half_t *, const half_t *, int, int, int);

template <typename T>
static int gemv_rowdot(const T *Mx, const T *x, T *y, const T *bias, int R, int K) {
    hipLaunchKernelGGL((gemv_rowdot_kernel<T, Traits<T>::VEC>), dim3((R + 3) / 4), dim3(256), 0, state().stream, Mx, x, y, bias, R, K);
    return hip_ok(hipGetLastError(), "gemv launch") ? 0 : 2;
}

template <typename T, int V>
static int gemv_coldot(const T *x, const T *Mx, T *y, int K, int M) {
    const GvShares sh = gv_shares<T, V>(K, M);
    hipLaunchKernelGGL((gemv_coldot_kernel<T, V>), dim3(sh.cols * sh.shares), dim3(GV_NT), 0, state().stream, x, Mx, y, K, M, sh);
    if (sh.shares > 1) launch_share_sum<T>(sh.part, y, M, sh.shares, state().stream);
    return hip_ok(hipGetLastError(), "gemv launch") ? 0 : 2;
}

// Whether C = A B^T takes the kernel that shares the contraction out over the waves of a 32 x 32 tile, in a grid of 17 to 8192
// samples, 8 to 8192 outputs and 16 to 1300 inputs (us, other routes / this): 1.3 times as fast in the mean of 233 fp32 layers,
// 1.2 of 189 in fp16.  As many tiles as the chip has compute units: contractions of at most four trips to memory (fp16 100 x 1024
// x 128 8.0 / 6.3, but from odd rows, which its scattered pieces cannot read at speed, 100 x 785 x 128 7.1 / 10.6; fp32 100 x 512 x
// 128 9.2 / 6.7, 100 x 785 x 333 10.6 / 8.0), fp32 up to 900, where its sums are as near to 64 bits as the other routes' (900:
// 1.19e-7 and 1.21e-7, 1153: 1.30e-7 and 1.18e-7).  Up to two tiles a compute unit, where the other routes have one launch of
// larger tiles: fp32 from rows that they cannot read in whole slabs up to 800 (714 16.6 / 13.9, 886 19.4 / 20.5), aligned ones
// of 512 to 600 (512 12.9 / 10.8, 240 9.0 / 8.9, 576 14.4 / 14.4, 832 18.0 / 18.9, 1152 15.5 / 22.8); fp16 up to 256 but for whole
// slabs (128 4.7 / 6.4, 192 5.0 / 6.6; 64 5.0 / 4.9).
template <typename T>
static bool deep_pays(const T *A, const T *B, int N, int M, int K) {
    constexpr int VEC = Traits<T>::VEC;
    const long long tiles = (long long)((N + 31) / 32) * ((M + 31) / 32), cu = state().num_cu;
    if (state().gemm_path != 0 || K < VEC || tiles > 2 * cu) return false;
    if (sizeof(T) == 4) return tiles <= cu ? K <= 900 : K % 16 ? K <= 800 : K >= 512 && K <= 600;
    return K % 2 == 0 && ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 3) == 0 &&
           (tiles <= cu ? K <= 1024 : K <= 256 && (K % 64 != 0 || K == 64));
}

template <typename T>
int mm_dispatch(const T *A, const T *B, T *C, int N, int M, int K, int trans_B, const T *bias) {
    if (!ensure_init()) return 2;
    state().last_gemm_form = 0;
    if (N <= 0 || M <= 0 || K <= 0) return 0;  // K == 0 leaves C untouched, as mm() does
    constexpr int VEC = Traits<T>::VEC;
    if (K == 1 && !bias) return M >= VEC ? outer<T, VEC>(A, B, C, N, M) : outer<T, 1>(A, B, C, N, M);
    if (M == 1 && !bias) return gemv_rowdot<T>(A, B, C, nullptr, N, K);  // B is K x 1 or 1 x K: the same vector
    if (N == 1 && trans_B) return gemv_rowdot<T>(B, A, C, bias, M, K);
    if (N == 1 && !bias) return M >= VEC ? gemv_coldot<T, VEC>(A, B, C, K, M) : gemv_coldot<T, 1>(A, B, C, K, M);
    if (trans_B && deep_pays<T>(A, B, N, M, K)) return ragged_deep<T>(A, B, C, N, M, K, bias);
    GemmArgs g = {};
    g.A = A;
    g.B = B;
    g.C = C;
    g.N = N;
    g.M = M;
    g.K = K;
    g.a.row = axis_plain(N, K);
    g.a.k = axis_plain(K, 1);
    g.a.HL = g.a.WL = 1;
    if (trans_B) {
        g.b.row = axis_plain(M, K);
        g.b.k = axis_plain(K, 1);
    } else {
        g.b.row = axis_plain(M, 1);
        g.b.k = axis_plain(K, M);
    }
    g.b.HL = g.b.WL = 1;
    g.c.n = axis_plain(N, M);
    g.c.m = axis_plain(M, 1);
    g.bias = bias;
    return gemm<T>(g);
}

template int mm_dispatch<float>(const float *, const float *, float *, int, int, int, int, const float *);
template int mm_dispatch<half_t>(const half_t *, const half_t *, half_t *, int, int, int, int, const half_t *);

}  // namespace ptl
