// Householder reflectors of the FP64 reductions (tridiag.hip, band.hip).
#pragma once

#include <hip/hip_runtime.h>

// Below this sum of squares (elements of at most 3e-145) squares are subnormal or
// zero: beta, tau and the scale would come from a few bits and I - tau u u^T would
// not be orthogonal.  Such columns (blocks of a matrix that hardly couple) are
// multiplied by kRescale, which brings every nonzero double between 5e-35 and
// 1e145, and beta by its inverse.
constexpr double kSquareMin = 0x1p-960, kRescale = 0x1p960;

// The reflector of x (alpha at the pivot, sigma the squares of the rest):
// H = I - tau u u^T, u = 1 at the pivot and x * scale elsewhere, H x = beta.
struct Reflector {
    double beta, tau, scale;
};
__device__ __forceinline__ Reflector reflector(double alpha, double sigma) {
    if (sigma == 0.0) return {alpha, 0.0, 0.0};
    const double beta = -copysign(sqrt(alpha * alpha + sigma), alpha);
    return {beta, (beta - alpha) / beta, 1.0 / (alpha - beta)};
}
