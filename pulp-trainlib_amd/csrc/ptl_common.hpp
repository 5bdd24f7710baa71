// Shared declarations of the HIP side: separable index maps, the GEMM
// problem descriptor, library state and error plumbing.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ptl {

typedef _Float16 half_t;

// Largest spatial extent the packed coordinate look-up entries can carry.
constexpr int HW_LIMIT = 8191;

// ---------------------------------------------------------------------------
// Separable three-digit index map.
//
// An index idx in [0, n) is split as idx = (q2*d1 + q1)*d0 + q0 and mapped to
//   off = q2*o2 + q1*o1 + q0*o0 + ob   (element offset into a tensor)
//   h   = q2*h2 + q1*h1 + q0*h0 + hb   (vertical coordinate contribution)
//   w   = q2*w2 + q1*w1 + q0*w0 + wb   (horizontal coordinate contribution)
// A GEMM operand element (row, k) lives at off(row) + off(k) and exists iff
// 0 <= h(row)+h(k) < HL and 0 <= w(row)+w(k) < WL; elements that do not exist
// read as zero.  Plain matrices, batched CHW/HWC tensors and the implicit
// im2col patch matrices of forward, weight-gradient and input-gradient
// convolution are all instances of this form.
// ---------------------------------------------------------------------------
struct AxisMap {
    int n;           // extent
    int d1, d0;      // digit radices
    int o2, o1, o0, ob;
    int h2, h1, h0, hb;
    int w2, w1, w0, wb;
};

// How an operand tile is fetched from global memory.
enum FillMode : int {
    FILL_ELEM_K = 0,  // element loads, consecutive threads along k
    FILL_ELEM_R = 1,  // element loads, consecutive threads along rows
    FILL_VEC_K = 2,   // 16-byte loads along k   (k is a plain contiguous axis)
    FILL_VEC_R = 3,   // 16-byte loads along rows (row is a contiguous axis)
};

struct OperandMap {
    AxisMap row;
    AxisMap k;
    int HL, WL;  // coordinate box
    int mode;    // FillMode
};

struct OutMap {
    AxisMap n;
    AxisMap m;
};

struct GemmArgs {
    const void *A;
    const void *B;
    void *C;       // output tensor (written through `c` when splits == 1)
    float *ws;     // split-K partial sums, [splits][N][M] fp32
    const void *bias;  // added per m where the product is stored (not by the register-staged kernel)
    OperandMap a;  // rows = n index
    OperandMap b;  // rows = m index
    OutMap c;
    int N, M, K;
    int splits;
    int kchunk;    // K range per split (multiple of the k tile)
    int tiles_n, tiles_m;
    // Convolution as a sum over filter taps (look-up-free kernel only): k runs over (tap, channel); after the
    // `slabs_per_tap` slabs of a tap the A pointer jumps to the next tap of the padded, channel-blocked input:
    // by tap_jump_x bytes within a filter row, by tap_jump_y at the end of one.  taps <= 1: an ordinary product.
    // Lean kernel, k in runs: after every seg_slabs slabs the slab pointers of A / B jump by these bytes (k
    // made of an outer digit and a contiguous inner one, e.g. (sample, pixel)); 0 = k is one run.
    int seg_slabs;
    long long a_seg_jump, b_seg_jump;
    int taps, slabs_per_tap, tap_kw;
    long long tap_jump_x, tap_jump_y;
    // Weight gradient over taps: grid.y enumerates (tap, k split), tap_splits splits per tap; tap (ky, kx) reads
    // B shifted by ky*tap_jump_y + kx*tap_jump_x bytes and writes its own partial sums.  0: off.
    int tap_splits;
};

inline AxisMap axis_plain(int n, int stride, int base = 0) {
    AxisMap a = {};
    a.n = n;
    a.d1 = 1;
    a.d0 = n > 0 ? n : 1;
    a.o0 = stride;
    a.ob = base;
    return a;
}

// idx = q1*d0 + q0 with independent strides (e.g. (sample, pixel)).
inline AxisMap axis_two(int n, int d0, int s1, int s0, int base = 0) {
    AxisMap a = {};
    a.n = n;
    a.d1 = 1 << 30;
    a.d0 = d0;
    a.o1 = s1;
    a.o0 = s0;
    a.ob = base;
    return a;
}

__host__ __device__ inline void axis_decode(const AxisMap &a, int idx, int &off, int &h, int &w) {
    // One- and two-digit maps are the common case; skip the divisions they do not need
    // (the branches are uniform across a wave).
    int q0, q1, q2;
    if (a.d0 >= a.n) {
        q0 = idx;
        q1 = 0;
        q2 = 0;
    } else if (a.d1 >= (1 << 30)) {
        q1 = idx / a.d0;
        q0 = idx - q1 * a.d0;
        q2 = 0;
    } else {
        int t = idx / a.d0;
        q0 = idx - t * a.d0;
        q2 = t / a.d1;
        q1 = t - q2 * a.d1;
    }
    off = q2 * a.o2 + q1 * a.o1 + q0 * a.o0 + a.ob;
    h = q2 * a.h2 + q1 * a.h1 + q0 * a.h0 + a.hb;
    w = q2 * a.w2 + q1 * a.w1 + q0 * a.w0 + a.wb;
}

// ---------------------------------------------------------------------------
// Library state
// ---------------------------------------------------------------------------
struct State {
    bool ready = false;
    int device = -1;
    hipStream_t stream = nullptr;
    float *ws = nullptr;  // split-K / partial-sum workspace
    size_t ws_bytes = 0;
    void *scratch = nullptr;  // general scratch (dilated gradients, staging)
    size_t scratch_bytes = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int num_cu = 256;
    void *zeros = nullptr;  // 256 zero bytes: source of elements that do not exist
    int gemm_path = 0;      // 0: fastest kernel that fits; 1: staged GEMM only; others: one route wherever it fits (see ptl_set_gemm_path)
    int last_gemm_streamed = 0;  // 1 if the last pipelined GEMM ran the streaming kernel
    int last_conv_resident = 0;  // 1 if the last Conv2D forward / input-gradient call kept its input tile in LDS for all taps
    int last_conv_direct = 0;  // 1 if the last Conv2D forward / input-gradient call ran the direct kernel
    int last_gemm_tile = 0;    // rows * 1000 + columns of the tile of the last look-up-free pipelined product
    int staging_copies = 0;  // see ptl_staging_copies
    int last_gemm_form = 0;    // of the last dense layer, matrix product, Conv2D or attention call: see ptl_last_gemm_form
};

State &state();
bool ensure_init();
void set_error(const char *fmt, ...);
bool hip_ok(hipError_t e, const char *what);
float *workspace(size_t bytes);
float *workspace_if(size_t bytes);  // nullptr, and no error, where it would have to grow and cannot: in a capture, for lack of memory
void *scratch(size_t bytes);

template <typename T>
int gemm(const GemmArgs &g);  // returns 0 on success

// Pipelined LDS-DMA kernel: 0 = launched, -1 = problem does not fit, 2 = HIP failure.
template <typename T>
int gemm_async(GemmArgs &g);

// Two independent products; one launch where both fit the look-up-free kernel with the same
// tile shape, else one after the other.
template <typename T>
int gemm_pair(const GemmArgs &g0, const GemmArgs &g1);
// The one launch alone: -1 when the products do not share one.
template <typename T>
int gemm_pair_lean(const GemmArgs &g0, const GemmArgs &g1);
// Weight, input and (where db is given) bias gradient of a dense layer in one launch: on one sample; on a batch.
template <typename T>
int linear_one_bw(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int in, int out);
// ... and on two to LINEAR_FEW; the forward pass of two to sixteen.
constexpr int LINEAR_FEW = 8;
template <typename T>
int linear_few_bw(const T *x, const T *W, const T *dy, T *dW, T *dx, T *db, int ns, int in, int out);
template <typename T>
int linear_few_fw(const T *x, const T *W, T *y, const T *bias, int ns, int in, int out);
template <typename T>
int linear_bw_ragged(const T *X, const T *W, const T *dY, T *dW, T *dX, T *db, int ns, int in, int out);
template <typename T>
int gemm_async_pair(GemmArgs &g0, GemmArgs &g1);

// GEMV / outer-product kernels for products with a unit dimension.  `bias` (per column) is added where it is given.
template <typename T>
int mm_dispatch(const T *A, const T *B, T *C, int N, int M, int K, int trans_B, const T *bias = nullptr);

#ifdef __HIP_DEVICE_COMPILE__
// Asks for lines of a kernel's arguments together.  They lie in memory and the compiler loads each where it is needed: a line
// that is asked for behind an index or a branch that came from another line is one more trip, of about 1000 clocks, before
// the first load of data.  Worth it where there are many lines or trips: products of any size, whose arguments are 300 to 4000
// bytes (9 samples, 22 -> 8 channels, 13 x 13, 3 x 3 in fp16, forward and backward 23.1 -> 20.8 us; 200 drawn passes 1.02 in the mean,
// convolutions 1.04), patch rows, transpositions.  In row dots, batch norms, tiled convolutions and sums it gave nothing
// that could be measured, and lines that a workgroup does not need cost (all five products' for a pair: 24.2 -> 24.8 us).
template <typename... A>
constexpr int args_bytes() {
    int n = 0;
    ((n = (n + (int)alignof(A) - 1) / (int)alignof(A) * (int)alignof(A) + (int)sizeof(A)), ...);
    return n;
}
// B0 bytes from a0 on, B1 from a1 and B2 from a2: whole words.
template <int B0, int B1 = 0, int B2 = 0>
__device__ __forceinline__ void fetch_args_at(int a0, int a1 = 0, int a2 = 0) {
    typedef const char __attribute__((address_space(4))) *Bytes;
    const Bytes p = (Bytes)__builtin_amdgcn_kernarg_segment_ptr();
    unsigned word;
    asm volatile(
        ".macro ptl_fetch base, lines, last\n"
        ".set ptl_arg, 0\n"
        ".rept \\lines\n"
        "s_load_dword %0, \\base, ptl_arg\n"
        ".set ptl_arg, ptl_arg + 64\n"
        ".endr\n"
        "s_load_dword %0, \\base, \\last\n"
        ".endm\n"
        "ptl_fetch %1, %c4, %c7\n"
        ".if %c5\n"
        "ptl_fetch %2, %c5, %c8\n"
        ".endif\n"
        ".if %c6\n"
        "ptl_fetch %3, %c6, %c9\n"
        ".endif\n"
        ".purgem ptl_fetch\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(word)
        : "s"(p + a0), "s"(p + a1), "s"(p + a2), "i"((B0 + 63) / 64), "i"((B1 + 63) / 64), "i"((B2 + 63) / 64), "i"(B0 - 4), "i"(B1 - 4), "i"(B2 - 4)
        : "memory");
}
template <typename... A>
__device__ __forceinline__ void fetch_args(const A &...) {  // all arguments, in their order
    fetch_args_at<args_bytes<A...>()>(0);
}
#else
template <int, int = 0, int = 0>
__device__ inline void fetch_args_at(int, int = 0, int = 0) {}
template <typename... A>
__device__ inline void fetch_args(const A &...) {}
#endif

}  // namespace ptl
