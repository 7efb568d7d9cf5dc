// Per-pixel term of the residual pass (odie/residual_cuda.cu:20-33, odie/selection.py:58-73):
// t = byte / 255 (correctly rounded fp32 division) or the fp32 target, d = p - t in fp32,
// rgb = (double(d0*d0) + double(d1*d1)) + double(d2*d2), term = rgb / 3.0 in fp64.  Shared by
// the streamed residual (residual.hip) and the fused reconstruction (reconstruct.hip).
#pragma once
#include "common.h"

namespace odie {

// Correctly rounded quotients by a constant d from its rounded reciprocal r: with q = fl(x r) and
// the exact remainder x - q d, fl(q + r (x - q d)) is the rounded quotient (Markstein, "Computation
// of elementary functions on the IBM RISC System/6000 processor", 1990) where nothing underflows,
// three operations in place of the ten of a general division; an infinite or NaN x leaves a NaN
// remainder, and then q itself is the quotient.  byte / 255 is checked for all 256 bytes; the
// squares of fp32 differences are zero or at least 2^-149, so x / 3 stays far from underflow.
__device__ inline float byte_target(uint8_t value) {
    constexpr float kReciprocal = 1.0f / 255.0f;
    const float x = static_cast<float>(value), q = x * kReciprocal;
    return __builtin_fmaf(__builtin_fmaf(-255.0f, q, x), kReciprocal, q);
}

__device__ inline double third(double x) {
    constexpr double kReciprocal = 1.0 / 3.0;
    const double q = x * kReciprocal;
    const double remainder = __builtin_fma(-3.0, q, x);
    return remainder == remainder ? __builtin_fma(remainder, kReciprocal, q) : q;
}

__device__ inline double residual_term(float p0, float p1, float p2, float t0, float t1, float t2) {
    const float d0 = p0 - t0, d1 = p1 - t1, d2 = p2 - t2;
    double rgb = static_cast<double>(d0 * d0) + static_cast<double>(d1 * d1);
    rgb = rgb + static_cast<double>(d2 * d2);
    return third(rgb);
}

}  // namespace odie
