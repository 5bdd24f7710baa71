// Library state, error reporting, workspace and host-pointer staging.
#include "ptl_common.hpp"
#include "ptl_host.hpp"

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace ptl {

static thread_local char g_err[512] = "";
static thread_local int g_status = 0;

State &state() {
    static State s;
    return s;
}

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

const char *last_error() { return g_err; }
int last_status() { return g_status; }
void set_status(int s) {
    g_status = s;
    if (s != 0) fflush(stdout);  // make the rejection message visible right away
}

bool hip_ok(hipError_t e, const char *what) {
    if (e == hipSuccess) return true;
    set_error("%s: %s", what, hipGetErrorString(e));
    return false;
}

int init_device(int device) {
    State &st = state();
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count == 0) {
        (void)hipGetLastError();
        set_error("libptl_hip: no HIP device available (%s); there is no CPU fallback",
                  e == hipSuccess ? "device count is 0" : hipGetErrorString(e));
        return 2;
    }
    if (device < 0 || device >= count) {
        set_error("libptl_hip: device %d out of range (0..%d)", device, count - 1);
        return 1;
    }
    if (!hip_ok(hipSetDevice(device), "hipSetDevice")) return 2;
    if (st.ready && st.device == device) return 0;
    hipDeviceProp_t prop;
    if (!hip_ok(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties")) return 2;
    st.num_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    if (!st.ev0) {
        if (!hip_ok(hipEventCreate(&st.ev0), "hipEventCreate")) return 2;
        if (!hip_ok(hipEventCreate(&st.ev1), "hipEventCreate")) return 2;
    }
    if (!st.zeros) {
        if (!hip_ok(hipMalloc(&st.zeros, 256), "hipMalloc(zeros)")) return 2;
        if (!hip_ok(hipMemset(st.zeros, 0, 256), "hipMemset(zeros)")) return 2;
    }
    if (int rc = dw_noalloc_setup(device)) return rc;
    st.device = device;
    st.ready = true;
    return 0;
}

bool ensure_init() {
    State &st = state();
    if (st.ready) return true;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        dev = 0;
    }
    return init_device(dev) == 0;
}

// True while the library's stream records into a HIP graph: synchronising, freeing and allocating are illegal then
// (each of them would invalidate the capture).
static bool stream_is_capturing(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &status) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return status != hipStreamCaptureStatusNone;
}

static size_t grown(size_t want) { return want < (size_t)(8u << 20) ? (size_t)(8u << 20) : want + want / 4; }

static void *grow(void *&buf, size_t &have, size_t want, const char *what) {
    if (want <= have) return buf;
    State &st = state();
    if (stream_is_capturing(st.stream)) {
        set_error("%s: %zu bytes are needed and %zu are there, and the stream is being captured into a graph; call "
                  "ptl_reserve() or run this shape once before the capture begins", what, want, have);
        return nullptr;
    }
    if (buf) {
        // kernels enqueued earlier - on this stream or on one the caller selected before - may still read the
        // old buffer
        if (!hip_ok(hipDeviceSynchronize(), "hipDeviceSynchronize")) return nullptr;
        (void)hipFree(buf);
        buf = nullptr;
        have = 0;
    }
    const size_t sz = grown(want);
    if (!hip_ok(hipMalloc(&buf, sz), what)) {
        buf = nullptr;
        return nullptr;
    }
    have = sz;
    return buf;
}

float *workspace(size_t bytes) {
    State &st = state();
    void *p = st.ws;
    void *got = grow(p, st.ws_bytes, bytes, "hipMalloc(workspace)");
    st.ws = static_cast<float *>(p);  // (a growth that is refused leaves the one that is there)
    return static_cast<float *>(got);
}

// For a caller that has another way without it.  The larger buffer comes before the present one goes, so that a refusal costs neither
// that one nor a wait; only a lack of memory is passed over, another HIP error is left for the launch behind to report.
float *workspace_if(size_t bytes) {
    State &st = state();
    if (bytes <= st.ws_bytes) return st.ws;
    if (stream_is_capturing(st.stream)) return nullptr;
    const size_t sz = grown(bytes);
    void *more = nullptr;
    const hipError_t e = hipMalloc(&more, sz);
    if (e != hipSuccess) {
        if (e == hipErrorOutOfMemory) (void)hipGetLastError();
        return nullptr;
    }
    if (st.ws) {
        if (hipDeviceSynchronize() != hipSuccess) {  // (see grow())
            (void)hipFree(more);
            return nullptr;
        }
        (void)hipFree(st.ws);
    }
    st.ws = static_cast<float *>(more);
    st.ws_bytes = sz;
    return st.ws;
}

void *scratch(size_t bytes) {
    State &st = state();
    return grow(st.scratch, st.scratch_bytes, bytes, "hipMalloc(scratch)");
}

// ---------------------------------------------------------------------------
// Staging of host pointers
// ---------------------------------------------------------------------------
static bool is_device_ptr(const void *p) {
    hipPointerAttribute_t attr;
    memset(&attr, 0, sizeof(attr));
    hipError_t e = hipPointerGetAttributes(&attr, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // plain host memory is reported as an error on some runtimes
        return false;
    }
    return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged;
}

// Device buffers for staged host tensors are kept between calls: a call that stages the same sizes again (a
// training loop on host arrays) allocates nothing.  A buffer is handed out again only after the call that used
// it has synchronised its stream (finish(), or the destructor of a Stager that never got there).
struct StagePool {
    struct Buf {
        void *dev;
        size_t bytes;
        bool busy;
    };
    std::mutex lock;
    std::vector<Buf> bufs;
    std::vector<StageBlock *> blocks;  // the idle ones, the one given back last at the end
    size_t total = 0, idle = 0;        // bytes of bufs, of blocks
};
static const size_t STAGE_POOL_LIMIT = (size_t)1 << 30;  // idle buffers beyond this are freed on release

// Tensors up to STAGE_SMALL bytes travel through a block.  A copy of its own costs a tensor about 10 us whatever its
// size (pageable memory: the runtime's own bounce buffer, a blit and a wait for it); through the block it costs the
// CPU's copy (8 us for 1 MB) and its share of two kernels of 3-5 us, which move 20-50 GB/s over the bus.
static const size_t STAGE_SMALL = (size_t)1 << 20;
static const size_t STAGE_BLOCK = (size_t)4 << 20;
// Larger ones, up to STAGE_LARGE bytes, take a block of their own and travel in STAGE_CHUNK parts: the bus moves one part
// while the CPU copies the next (on the way back: the one before).  Conv2D 32 -> 129 of 56 x 56, four
// samples in fp32, forward + backward (10 MB in, 9 MB out): 925 -> 850 us, the CPU's copies being most of what is left.
// What is larger still, or more than STAGE_CALL bytes in a call, is left to the runtime's copies of pageable memory.
static const size_t STAGE_LARGE = (size_t)32 << 20;
static const size_t STAGE_CHUNK = (size_t)1 << 20;
static const size_t STAGE_CALL = (size_t)128 << 20;
static const size_t STAGE_IDLE_LIMIT = (size_t)128 << 20;  // of idle blocks; beyond, the oldest are freed
static const int STAGE_EVENTS = (int)(STAGE_LARGE / STAGE_CHUNK);

struct StageBlock {
    char *host;  // pinned, mapped
    char *dev;
    size_t bytes;
    int device;  // that dev and the events belong to
    hipEvent_t done[STAGE_EVENTS];  // of the parts on their way back (made as they are needed)
};

static StagePool &stage_pool() {
    static StagePool p;
    return p;
}

static void block_free(StageBlock *b) {
    for (hipEvent_t e : b->done)
        if (e) (void)hipEventDestroy(e);
    if (b->host) (void)hipHostFree(b->host);
    if (b->dev) (void)hipFree(b->dev);
    delete b;
}

// A block of at least `bytes` (at most twice that: blocks are powers of two).
static StageBlock *block_acquire(size_t bytes) {
    const int device = state().device;
    size_t size = STAGE_CHUNK;
    while (size < bytes) size *= 2;
    StagePool &p = stage_pool();
    {
        std::lock_guard<std::mutex> g(p.lock);
        for (size_t i = p.blocks.size(); i-- > 0;)
            if (p.blocks[i]->bytes == size && p.blocks[i]->device == device) {
                StageBlock *b = p.blocks[i];
                p.blocks.erase(p.blocks.begin() + i);
                p.idle -= size;
                return b;
            }
    }
    StageBlock *b = new StageBlock{};
    b->bytes = size;
    b->device = device;
    if (hipHostMalloc(reinterpret_cast<void **>(&b->host), size, hipHostMallocDefault) != hipSuccess ||
        hipMalloc(reinterpret_cast<void **>(&b->dev), size) != hipSuccess) {
        (void)hipGetLastError();
        block_free(b);
        return nullptr;  // (the tensors take buffers of their own)
    }
    return b;
}

static void block_release(StageBlock *b) {
    StagePool &p = stage_pool();
    std::vector<StageBlock *> old;
    {
        std::lock_guard<std::mutex> g(p.lock);
        p.blocks.push_back(b);
        p.idle += b->bytes;
        while (p.idle > STAGE_IDLE_LIMIT) {
            old.push_back(p.blocks.front());
            p.idle -= p.blocks.front()->bytes;
            p.blocks.erase(p.blocks.begin());
        }
    }
    for (StageBlock *o : old) block_free(o);
}

static void *stage_acquire(size_t bytes) {
    StagePool &p = stage_pool();
    std::lock_guard<std::mutex> g(p.lock);
    int best = -1;
    for (size_t i = 0; i < p.bufs.size(); ++i) {
        const StagePool::Buf &b = p.bufs[i];
        if (b.busy || b.bytes < bytes || b.bytes > 2 * bytes + (1u << 20)) continue;
        if (best < 0 || b.bytes < p.bufs[best].bytes) best = (int)i;
    }
    if (best >= 0) {
        p.bufs[best].busy = true;
        return p.bufs[best].dev;
    }
    void *dev = nullptr;
    if (!hip_ok(hipMalloc(&dev, bytes), "hipMalloc(staging)")) return nullptr;
    p.bufs.push_back({dev, bytes, true});
    p.total += bytes;
    return dev;
}

static void stage_release(void *dev) {
    StagePool &p = stage_pool();
    std::lock_guard<std::mutex> g(p.lock);
    for (auto &b : p.bufs)
        if (b.dev == dev) b.busy = false;
    // keep the pool bounded: drop idle buffers, largest first
    while (p.total > STAGE_POOL_LIMIT) {
        int big = -1;
        for (size_t i = 0; i < p.bufs.size(); ++i)
            if (!p.bufs[i].busy && (big < 0 || p.bufs[i].bytes > p.bufs[big].bytes)) big = (int)i;
        if (big < 0) break;
        (void)hipFree(p.bufs[big].dev);
        p.total -= p.bufs[big].bytes;
        p.bufs.erase(p.bufs.begin() + big);
    }
}

// The staged tensors of one direction, in 16-byte pieces: piece i of segment s goes from src + at[s] + i to the same
// place in dst.  One side is pinned host memory: what bounds the kernel is the bus, so every thread has one piece in
// flight and the grid covers all of them (0.2 MB: 5 us against 5 copies of about 10 us each).
constexpr int STAGE_SEGS = 16;
struct StageCopy {
    const uint4 *src;
    uint4 *dst;
    unsigned at[STAGE_SEGS], first[STAGE_SEGS + 1];
    int n;
};
__global__ __launch_bounds__(256) void stage_copy_kernel(const StageCopy c) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= c.first[c.n]) return;
    int s = 0;
    while (s + 1 < c.n && i >= c.first[s + 1]) ++s;
    const unsigned p = c.at[s] + (i - c.first[s]);
    c.dst[p] = c.src[p];
}

static bool copy_part(uint4 *dst, const uint4 *src, size_t at, size_t bytes) {
    StageCopy c = {};
    c.src = src;
    c.dst = dst;
    c.n = 1;
    c.at[0] = (unsigned)(at / 16);
    c.first[1] = (unsigned)((bytes + 15) / 16);
    hipLaunchKernelGGL(stage_copy_kernel, dim3((c.first[1] + 255) / 256), dim3(256), 0, state().stream, c);
    return hip_ok(hipGetLastError(), "staging launch");
}

// A tensor with a block of its own: in part by part.
static bool block_send(StageBlock *b, const void *host, size_t bytes) {
    for (size_t at = 0; at < bytes; at += STAGE_CHUNK) {
        const size_t n = std::min(STAGE_CHUNK, bytes - at);
        memcpy(b->host + at, static_cast<const char *>(host) + at, n);
        if (!copy_part(reinterpret_cast<uint4 *>(b->dev), reinterpret_cast<const uint4 *>(b->host), at, n)) return false;
    }
    return true;
}
// Back: the copies are enqueued with an event behind each part, ...
static bool block_return(StageBlock *b, size_t bytes) {
    for (size_t at = 0, i = 0; at < bytes; at += STAGE_CHUNK, ++i) {
        const size_t n = std::min(STAGE_CHUNK, bytes - at);
        if (!copy_part(reinterpret_cast<uint4 *>(b->host), reinterpret_cast<const uint4 *>(b->dev), at, n)) return false;
        if (!b->done[i] && !hip_ok(hipEventCreateWithFlags(&b->done[i], hipEventDisableTiming), "hipEventCreate")) return false;
        if (!hip_ok(hipEventRecord(b->done[i], state().stream), "hipEventRecord")) return false;
    }
    return true;
}
// ... and each part is copied out as it arrives.
static bool block_receive(StageBlock *b, void *host, size_t bytes) {
    for (size_t at = 0, i = 0; at < bytes; at += STAGE_CHUNK, ++i) {
        if (!hip_ok(hipEventSynchronize(b->done[i]), "hipEventSynchronize")) return false;
        memcpy(static_cast<char *>(host) + at, b->host + at, std::min(STAGE_CHUNK, bytes - at));
    }
    return true;
}

// Enqueues the copies of the shared block's tensors that are pending (in) or to be returned (out).
bool Stager::launch_block_copy(bool in) {
    StageCopy c = {};
    c.src = reinterpret_cast<const uint4 *>(in ? block_->host : block_->dev);
    c.dst = reinterpret_cast<uint4 *>(in ? block_->dev : block_->host);
    auto flush = [&]() {
        if (c.n == 0) return true;
        hipLaunchKernelGGL(stage_copy_kernel, dim3((c.first[c.n] + 255) / 256), dim3(256), 0, state().stream, c);
        ++state().staging_copies;
        c.n = 0;
        return hip_ok(hipGetLastError(), "staging launch");
    };
    for (auto &t : items_) {
        if (t.own || !t.block || !(in ? t.pending : t.copy_out)) continue;
        t.pending = false;
        if (c.n == STAGE_SEGS && !flush()) return false;
        c.at[c.n] = (unsigned)((static_cast<char *>(t.dev) - block_->dev) / 16);
        c.first[c.n + 1] = c.first[c.n] + (unsigned)((t.bytes + 15) / 16);
        ++c.n;
    }
    return flush();
}

Stager *&Stager::scope() {
    static thread_local Stager *s = nullptr;
    return s;
}

bool Stager::failed() {
    Stager &r = root_ ? *root_ : *this;
    if (r.pending_ && !failed_) {
        r.pending_ = false;
        if (!r.launch_block_copy(true)) failed_ = true;
    }
    return failed_;
}

// What a step of a shared call wrote goes back to the caller, and is what later steps read, only if the step succeeded.
void Stager::keep_outputs(bool keep) {
    for (size_t i : marked_) (keep ? root_->items_[i].written : root_->items_[i].copy_out) = keep;
    marked_.clear();
}

void Stager::release() {
    for (auto &t : items_) {
        if (t.own) block_release(t.block);
        else if (t.dev && !t.block) stage_release(t.dev);
    }
    items_.clear();
    if (block_) block_release(block_);
    block_ = nullptr;
    block_used_ = own_bytes_ = 0;
    pending_ = false;
}

Stager::~Stager() {
    if (root_) keep_outputs(false);
    if (items_.empty()) return;
    // copies or kernels of a call that bailed out early may still be in flight on the buffers
    if (!finished_) (void)hipStreamSynchronize(state().stream);
    release();
}

void *Stager::map(const void *host_or_dev, size_t bytes, bool copy_in, bool copy_out) {
    if (failed_) return nullptr;
    if (!host_or_dev) {
        set_error("null tensor pointer");
        failed_ = rejected_ = true;
        return nullptr;
    }
    if (bytes == 0) return const_cast<void *>(host_or_dev);
    if (is_device_ptr(host_or_dev)) return const_cast<void *>(host_or_dev);
    if (device_only_) {
        set_error("host pointer passed to an entry point that may not allocate (staging needs device buffers)");
        failed_ = rejected_ = true;
        return nullptr;
    }
    Stager &r = root_ ? *root_ : *this;
    Item *hit = nullptr;
    for (auto &t : r.items_)
        if (t.host == host_or_dev && t.bytes >= bytes) hit = &t;
    if (!hit) {
        Item it = {};
        it.host = const_cast<void *>(host_or_dev);
        it.bytes = bytes;
        const size_t slot = (bytes + 255) / 256 * 256;
        if (bytes <= STAGE_SMALL && r.block_used_ + slot <= STAGE_BLOCK && (r.block_ || (r.block_ = block_acquire(STAGE_BLOCK)))) {
            it.block = r.block_;
            it.dev = r.block_->dev + r.block_used_;
            r.block_used_ += slot;
        } else if (bytes > STAGE_SMALL && bytes <= STAGE_LARGE && r.own_bytes_ + bytes <= STAGE_CALL && (it.block = block_acquire(bytes))) {
            it.own = true;
            it.dev = it.block->dev;
            r.own_bytes_ += bytes;
        } else {
            it.dev = stage_acquire(bytes);
        }
        if (!it.dev) {
            failed_ = true;
            return nullptr;
        }
        r.items_.push_back(it);
        hit = &r.items_.back();
    }
    if (copy_out && !hit->copy_out) {
        hit->copy_out = true;
        if (root_) marked_.push_back((size_t)(hit - r.items_.data()));
    }
    // a tensor first mapped as an output and later as an input of the same step still gets its contents
    if (copy_in && !hit->copied_in && !hit->written) {
        if (hit->own) {
            if (!block_send(hit->block, host_or_dev, hit->bytes)) {
                failed_ = true;
                return nullptr;
            }
            ++state().staging_copies;
        } else if (hit->block) {
            memcpy(r.block_->host + (static_cast<char *>(hit->dev) - r.block_->dev), host_or_dev, hit->bytes);
            hit->pending = r.pending_ = true;
        } else if (!hip_ok(hipMemcpyAsync(hit->dev, host_or_dev, hit->bytes, hipMemcpyHostToDevice, state().stream),
                           "hipMemcpy(H2D)")) {
            failed_ = true;
            return nullptr;
        } else {
            ++state().staging_copies;
        }
        hit->copied_in = true;
    }
    return hit->dev;
}

void Stager::discard() {
    if (root_) keep_outputs(false);
    if (items_.empty()) return;
    // copies into the buffers may still be in flight
    (void)hipStreamSynchronize(state().stream);
    release();
}

int Stager::finish(int rc) {
    if (root_) {
        keep_outputs(!failed_ && rc == 0);
        return failed_ ? 2 : rc;
    }
    if (items_.empty()) return failed_ ? 2 : rc;
    State &st = state();
    const bool back = !failed_ && rc == 0;
    if (back) {
        if (block_ && !launch_block_copy(false)) failed_ = true;
        for (auto &t : items_)
            if (t.copy_out && t.own && !block_return(t.block, t.bytes)) failed_ = true;
        for (auto &t : items_)
            if (t.copy_out && t.own && !failed_ && !block_receive(t.block, t.host, t.bytes)) failed_ = true;
        for (auto &t : items_)
            if (t.copy_out && !t.block) {
                if (!hip_ok(hipMemcpyAsync(t.host, t.dev, t.bytes, hipMemcpyDeviceToHost, st.stream),
                            "hipMemcpy(D2H)"))
                    failed_ = true;
            }
    }
    if (!hip_ok(hipStreamSynchronize(st.stream), "hipStreamSynchronize")) failed_ = true;
    else finished_ = true;
    if (back && !failed_)
        for (auto &t : items_)
            if (t.copy_out && t.block && !t.own) memcpy(t.host, block_->host + (static_cast<char *>(t.dev) - block_->dev), t.bytes);
    return failed_ ? 2 : rc;
}

}  // namespace ptl

extern "C" {

// The steps of one call between these two share their staged tensors (one copy in, one wait); end returns the call's
// status: that of the steps, or 2 if the results could not be returned.
static thread_local int g_call_depth = 0;
void ptl_internal_stage_begin(void) {
    if (g_call_depth++ == 0) ptl::Stager::scope() = new ptl::Stager;
}
int ptl_internal_stage_end(int rc) {
    if (--g_call_depth > 0) return rc;
    ptl::Stager *s = ptl::Stager::scope();
    ptl::Stager::scope() = nullptr;
    const int back = s->finish(0);
    delete s;
    return rc ? rc : back;
}

int ptl_init(int device) { return ptl::init_device(device); }
const char *ptl_last_error(void) { return ptl::last_error(); }
int ptl_last_status(void) { return ptl::last_status(); }
// Work already enqueued on the stream being left may still use the library's workspace; the next call would
// write it from the new stream, so the old stream is drained first (a no-op when it is idle).  A stream that is
// being captured cannot be drained: the switch is refused then (status 1, the stream stays), and a drain that
// fails (a destroyed handle) is reported the same way after the switch.
void ptl_set_stream(void *s) {
    ptl::State &st = ptl::state();
    hipStream_t next = static_cast<hipStream_t>(s);
    ptl::set_status(0);
    if (st.ready && next != st.stream) {
        if (ptl::stream_is_capturing(st.stream)) {
            ptl::set_error("ptl_set_stream: the current stream is being captured into a graph; switch streams "
                           "before the capture begins or after it ends");
            ptl::set_status(1);
            return;
        }
        hipError_t e = hipStreamSynchronize(st.stream);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            ptl::set_error("ptl_set_stream: draining the previous stream failed (%s)", hipGetErrorString(e));
            ptl::set_status(2);
        }
    }
    st.stream = next;
}

// Grows the two internal buffers (partial sums; blocked / padded copies) to at least the given sizes now, so that
// no later call has to: callers that capture the library's launches into a graph, or that may not allocate in
// their steady state, reserve once after ptl_init.  ptl_reserved reports the present sizes (after a warm-up pass
// over the caller's shapes they are the sizes those shapes need).
int ptl_reserve(size_t workspace_bytes, size_t scratch_bytes) {
    if (!ptl::ensure_init()) return 2;
    if (workspace_bytes && !ptl::workspace(workspace_bytes)) return 2;
    if (scratch_bytes && !ptl::scratch(scratch_bytes)) return 2;
    return 0;
}

void ptl_reserved(size_t *workspace_bytes, size_t *scratch_bytes) {
    ptl::State &st = ptl::state();
    if (workspace_bytes) *workspace_bytes = st.ws_bytes;
    if (scratch_bytes) *scratch_bytes = st.scratch_bytes;
}

void ptl_set_gemm_path(int path) { ptl::state().gemm_path = path; }
int ptl_last_conv_direct(void) { return ptl::state().last_conv_direct; }
int ptl_last_gemm_streamed(void) { return ptl::state().last_gemm_streamed; }
int ptl_last_conv_resident(void) { return ptl::state().last_conv_resident; }
int ptl_last_gemm_tile(void) { return ptl::state().last_gemm_tile; }
int ptl_last_gemm_form(void) { return ptl::state().last_gemm_form; }
int ptl_staging_copies(void) { return ptl::state().staging_copies; }

int ptl_sync(void) {
    if (!ptl::ensure_init()) return 2;
    return ptl::hip_ok(hipStreamSynchronize(ptl::state().stream), "hipStreamSynchronize") ? 0 : 2;
}

int ptl_timer_begin(void) {
    if (!ptl::ensure_init()) return 2;
    return ptl::hip_ok(hipEventRecord(ptl::state().ev0, ptl::state().stream), "hipEventRecord") ? 0 : 2;
}

float ptl_timer_end_ms(void) {
    if (!ptl::ensure_init()) return -1.f;
    ptl::State &st = ptl::state();
    if (!ptl::hip_ok(hipEventRecord(st.ev1, st.stream), "hipEventRecord")) return -1.f;
    if (!ptl::hip_ok(hipEventSynchronize(st.ev1), "hipEventSynchronize")) return -1.f;
    float ms = -1.f;
    if (!ptl::hip_ok(hipEventElapsedTime(&ms, st.ev0, st.ev1), "hipEventElapsedTime")) return -1.f;
    return ms;
}

}  // extern "C"
