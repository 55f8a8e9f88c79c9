// acc / d from r = 1 / d in FP64: the coarsest solves divide by the same diagonal (positive,
// finite) in each of their passes.
#pragma once
#include <cstdint>
#include <cstring>

namespace mael {

// FP32: the correctly rounded quotient where it is normal or 0. A quotient of two 24-bit numbers
// is at least 2^-49 of itself away from the middle between two of them, and the FP64 product
// is within 2^-52. A subnormal one can be that middle exactly, so it may come out wrong (it is
// subnormal then too, see subnormal_rank), except where d is one of 1 .. 6 (all were compared).
__host__ __device__ inline float quotient(float acc, float, double r) { return (float)((double)acc * r); }
// Less than SUBNORMALS for a subnormal q that is not 0 (q's magnitude as an integer, less 1).
constexpr uint32_t SUBNORMALS = 0x7fffff;
__host__ __device__ inline uint32_t subnormal_rank(float q) {
    uint32_t b;
    std::memcpy(&b, &q, sizeof b);
    return (b & 0x7fffffffu) - 1u;
}
// FP64, acc finite and neither the quotient nor its remainder subnormal: correctly rounded, by
// two Newton corrections, each with the exact remainder of a fused multiply-add.
__host__ __device__ inline double quotient(double acc, double d, double r) {
    double q = acc * r;
    q = __builtin_fma(__builtin_fma(-q, d, acc), r, q);
    return __builtin_fma(__builtin_fma(-q, d, acc), r, q);
}

}  // namespace mael
