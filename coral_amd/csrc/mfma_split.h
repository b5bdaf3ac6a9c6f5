// mfma_split.h -- fp32 rows as two planes of halves for the half-precision matrix cores (device code).
//
// A row x is scaled by a power of two that puts |x| into [2^13, 2^14); a scaled component is hi + lo with
// hi = half(x), lo = half(x - hi), where x - hi is exact: 22 bits of x.  An inner product of two rows is then
// hi.hi + hi.lo + lo.hi with exact products and fp32 accumulation.
//
// Error bound, with u = 2^-24.  Splitting: each component is off by at most 2^-22 of itself, and lo.lo is left out:
// 12 u |a| |b| over the sum (components below 2^-28 of their row's norm lose more, but of less: sqrt(dim) 2^-38 |a| |b|
// in all).  Accumulation: 3 dim additions, within 2 u of the running sum each even if the hardware truncates:
// 6 dim u |a| |b|.  Together (6 dim + 12) u |a| |b|.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace coral {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// e with |x| 2^e in [2^13, 2^14) for a row of squared norm n2; at most 60, which rows of norm 0 and of norms whose square
// leaves the normal range meet; at least kLeast.  -51 is what no finite norm falls below, so that no component of such a
// row leaves the range of a half and no product of two inverse scales overflows.  A row whose squared norm is infinite or
// NaN, or that a larger kLeast leaves with a component beyond 65 504, has hi = inf and lo = -inf there, and every product
// with it is NaN, which passes no comparison: callers must not take the absence of such a row for an answer.
template <int kLeast = -51>
__device__ __forceinline__ int mf_scale_exp(float n2) {
    const int E = (int)((__float_as_uint(n2) >> 23) & 0xffu) - 127;  // n2 in [2^E, 2^(E+1))
    return max(kLeast, min(60, 13 - (E >> 1)));
}
__device__ __forceinline__ float mf_pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// four scaled components as two planes of halves
__device__ __forceinline__ void mf_split4(const float4 a, float s, v4h& hi, v4h& lo) {
    const float x[4] = {a.x * s, a.y * s, a.z * s, a.w * s};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        hi[j] = (_Float16)x[j];
        lo[j] = (_Float16)(x[j] - (float)hi[j]);
    }
}

// eight scaled components as two planes of halves
__device__ __forceinline__ void mf_split8(const float4 a, const float4 b, float s, v8h& hi, v8h& lo) {
    const float x[8] = {a.x * s, a.y * s, a.z * s, a.w * s, b.x * s, b.y * s, b.z * s, b.w * s};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        hi[j] = (_Float16)x[j];
        lo[j] = (_Float16)(x[j] - (float)hi[j]);
    }
}

}  // namespace coral
