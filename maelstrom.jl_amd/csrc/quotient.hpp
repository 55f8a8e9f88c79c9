// acc / d, correctly rounded, from r = 1 / d in FP64: the coarsest solves divide by the same
// diagonal (finite, positive) in each of their passes.
#pragma once

namespace mael {

// FP32. For a normal result the FP64 product rounds to it: the quotient of two 24-bit numbers
// is at least 2^-49 of itself away from the middle between two of them, the product's error
// is under 2^-52. A subnormal one can be that middle exactly, so it takes the division.
__host__ __device__ inline float quotient(float acc, float d, double r) {
    const float q = (float)((double)acc * r);
    return __builtin_fabsf(q) >= 1.17549435e-38f || acc == 0.0f ? q : acc / d;
}
// FP64, acc finite and neither the quotient nor its remainder subnormal: two Newton
// corrections of the quotient, each with the exact remainder of a fused multiply-add.
__host__ __device__ inline double quotient(double acc, double d, double r) {
    double q = acc * r;
    q = __builtin_fma(__builtin_fma(-q, d, acc), r, q);
    return __builtin_fma(__builtin_fma(-q, d, acc), r, q);
}
// FP32 with d one of 1 .. 6: right for subnormal results too (every one of them was compared).
__host__ __device__ inline float quotient_small(float acc, double r) { return (float)((double)acc * r); }

}  // namespace mael
