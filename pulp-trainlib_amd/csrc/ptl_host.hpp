// Host-side helpers shared by the entry-point translation units.
#pragma once
#include "ptl_common.hpp"

#include <vector>

namespace ptl {

const char *last_error();
int last_status();
void set_status(int s);
int init_device(int device);
int dw_noalloc_setup(int device);  // looks up the fixed partial-sum array of the current device

// Whether two tensors (n elements of T each) share memory.  A launch that forms two gradients at once wants tensors that do
// not: where they do, the steps run one after the other, each complete before the next (an input gradient may be
// written over the input).
template <typename T>
inline bool share_memory(const T *a, size_t na, const T *b, size_t nb) {
    return a && b && a < b + nb && b < a + na;
}
// Of a backward call: the gradients dW, dX and db against what the call reads and against each other.
template <typename T>
inline bool backward_shares_memory(const T *X, size_t nx, const T *W, size_t nw, const T *dY, size_t ny, const T *dW, const T *dX,
                                   const T *db, size_t nb) {
    const T *in[3] = {X, W, dY}, *out[3] = {dX, dW, db};
    const size_t n_in[3] = {nx, nw, ny}, n_out[3] = {nx, nw, nb};
    for (int o = 0; o < 3; ++o) {
        for (int i = 0; i < 3; ++i)
            if (share_memory(out[o], n_out[o], in[i], n_in[i])) return true;
        if (share_memory(out[o], n_out[o], out[(o + 1) % 3], n_out[(o + 1) % 3])) return true;
    }
    return false;
}

struct StageBlock;  // pinned host memory and device memory of one size, from a pool (ptl_runtime.hip)

// Maps caller pointers to device pointers.  Device pointers pass through;
// host pointers get a device buffer from a pool kept between calls, filled
// before the kernels run (copy_in) and copied back by finish() (copy_out).
// finish() synchronises only when something was staged.
// Small host tensors share one pinned block: the CPU copies them into it as they are mapped, failed() - which every
// caller asks after its mappings and before its launches - enqueues one kernel that fetches all of them, and finish()
// one that writes all results back.  Larger ones have a pinned block each and move part by part, the CPU's copies beside
// the bus's.
class Stager {
   public:
    // device_only: host pointers are rejected instead of staged (callers that may not allocate)
    explicit Stager(bool device_only = false) : root_(scope()), device_only_(device_only) {}
    ~Stager();
    Stager(const Stager &) = delete;
    Stager &operator=(const Stager &) = delete;

    template <typename T>
    const T *in(const T *p, size_t n) {
        return static_cast<const T *>(map(p, n * sizeof(T), true, false));
    }
    template <typename T>
    T *out(T *p, size_t n) {
        return static_cast<T *>(map(p, n * sizeof(T), false, true));
    }
    template <typename T>
    T *inout(T *p, size_t n) {
        return static_cast<T *>(map(p, n * sizeof(T), true, true));
    }
    bool failed();  // enqueues the copies that are pending
    bool rejected() const { return rejected_; }  // failed because of the arguments, not because of HIP
    int finish(int rc);
    // Gives the staging buffers back without copying anything out (the kernels they were mapped for did not run).
    void discard();

    // The Stager that those made on this thread from now on share (NULL: each its own): a call made of several steps
    // fetches every host tensor once and waits once, at the end.  A step that fails still returns nothing.  What a step
    // has written is what the next one reads, at the same address; host tensors of a call that overlap in part are taken
    // for different ones.
    static Stager *&scope();

   private:
    struct Item {
        void *host;
        void *dev;
        size_t bytes;
        bool copy_out;
        bool copied_in;
        bool written;       // by a step that succeeded: the device's copy is the valid one
        bool own;           // block is this tensor's alone
        bool pending;       // in the pinned half of the shared block, to be fetched
        StageBlock *block;  // dev lies in it; NULL: a buffer of its own
    };
    void *map(const void *p, size_t bytes, bool copy_in, bool copy_out);
    bool launch_block_copy(bool in);
    void release();
    void keep_outputs(bool keep);
    std::vector<Item> items_;
    Stager *root_;
    std::vector<size_t> marked_;  // items of root_ that this step is the first to write
    StageBlock *block_ = nullptr;
    size_t block_used_ = 0, own_bytes_ = 0;
    bool pending_ = false;
    bool failed_ = false;
    bool finished_ = false;
    bool device_only_ = false;
    bool rejected_ = false;
};

}  // namespace ptl
