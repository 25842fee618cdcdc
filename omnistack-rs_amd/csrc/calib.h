// Shared by the two calibrations: calib.hip (samples stored by bins) and
// calib_inplace.hip (no copy of the samples).
#pragma once

#include "omni_common.h"

namespace omni {

constexpr int kLmK = 16;                    // centroids

// Arguments of omni_lloyd_max (checked).
struct LmCall {
    const void *x;
    int x_dtype, groups;
    int64_t outer, inner, outer_stride, group_stride;
    int max_iters;
    float tol;
    float *out;         // [g][16]
    int32_t *iters;     // [g], nullable
};

// The order-preserving key of an fp32 value, and back.
__device__ __forceinline__ uint32_t lm_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float lm_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

static inline size_t lm_align256(size_t x) { return (x + 255) & ~(size_t)255; }

// calib_inplace.hip
size_t lm_inplace_bytes(int groups, int64_t n);
void lm_inplace_run(const LmCall &c, void *workspace, hipStream_t st);

}  // namespace omni
