// cutoff.h -- which image Gaussians the residual pass of the two launches takes
// at a 64-pixel slot, and how.  Also compiled for the host, by its test.
#pragma once

#include <cmath>

#include "fpho_internal.h"

namespace fpho {

// the median of three numbers; 1 / v to one unit in the last place
FPHO_HDI float med3(float a, float b, float c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_fmed3f(a, b, c);
#else
    return std::fmax(std::fmin(a, b), std::fmin(std::fmax(a, b), c));
#endif
}
FPHO_HDI float reciprocal(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(v);
#else
    return 1.0f / v;
#endif
}

// Whether residual_kernel may test a Gaussian with meets() and visit it at pixels
// beyond its cutoff, where a pair then adds an exact zero: its centre lies within
// kPlainCoord of the exposure's origin, its F is positive definite with 1 - rho^2
// above kPlainRho, F is below 1.4e6 and the amplitude finite in FP32, so v' < 3e12
// and h' is finite at every pixel within kMaskedCoord.  (A NaN fails.)
// kPlainRho: a source of axis ratio 0.1, far larger than its PSF, has 4e-4; below,
// the FP32 error of rho takes the margin of meets() with it (an accepted pixel in
// a refused box about once in 10^5 boxes on the ellipse's edge at 1e-10).
constexpr double kPlainCoord = 262144.0;   // half an FP32 step below it: under 0.01 pixel
constexpr double kPlainRho = 1.0e-4;
constexpr uint32_t kNotPlain = 1;          // HotGauss::tag in the workspace
FPHO_HDI bool plain(double xcen, double ycen, double sfxx, double sfyy, double sfxy,
                    double ampA) {
    return std::fabs(xcen) < kPlainCoord && std::fabs(ycen) < kPlainCoord &&
           sfxx < 0.0 && sfxx > -1.0e6 && sfyy < 0.0 && sfyy > -1.0e6 &&
           sfxx * sfyy - sfxy * sfxy > kPlainRho * sfxx * sfyy &&
           std::fabs(ampA) < 3.0e38;
}

// For plain() Gaussians: false only if no pixel of the box [xlo, xhi] x [ylo, yhi]
// (relative to the centre) passes the cutoff test E <= 36.  The smallest E
// of a box that does not hold the centre is on an edge that faces the centre;
// along such an edge E is a parabola with its minimum at -(Fxy / Fyy) dx (or
// its twin).  sF is negative, so the smallest E is the largest E'.  The limit
// is widened by 0.1% and by the FP32 error of E, 4e-6 of it per 1 / (1 -
// rho^2), here and in pass 1.
FPHO_HDI bool meets(float xlo, float xhi, float ylo, float yhi, float sfxx,
                    float sfyy, float sfxy) {
    const float dx = med3(0.0f, xlo, xhi);
    const float dy = med3(0.0f, ylo, yhi);
    const float ya = med3(-sfxy * reciprocal(sfyy) * dx, ylo, yhi);
    const float xb = med3(-sfxy * reciprocal(sfxx) * dy, xlo, xhi);
    const float ea = fmaf(dx, fmaf(sfxx, dx, 2.0f * sfxy * ya), sfyy * ya * ya);
    const float eb = fmaf(dy, fmaf(sfyy, dy, 2.0f * sfxy * xb), sfxx * xb * xb);
    const float k = sfxx * sfyy;
    const float wide = k * reciprocal(fmaxf(fmaf(-sfxy, sfxy, k), 0.0f));
    return !(fmaxf(ea, eb) < kCutScaled * fmaf(4e-6f, wide, 1.001f));
}

}  // namespace fpho
