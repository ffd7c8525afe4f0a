// Random image Gaussians against random pixel boxes: every pixel that the FP32
// cutoff test of the pixel pass accepts has to lie in a box that the visit test
// (meets() for plain Gaussians, the cutoff box for the others) accepts.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <random>

#include "cutoff.h"

using namespace fpho;

namespace {

struct Trial {
    double xc, yc, a, b, d;   // centre, covariance [[a, b], [b, d]]
};

// pass 1's exponent at a pixel (fused forms as in the kernels)
bool inside(float x, float y, float xcen, float ycen, float xlo, float ylo, bool centre,
            float sfxx, float sfyy, float sfxy) {
    float dx = x - xcen, dy = y - ycen;
    if (centre) {
        dx -= xlo;
        dy -= ylo;
    }
    const float vx = std::fma(sfxx, dx, sfxy * dy);
    const float vy = std::fma(sfyy, dy, sfxy * dx);
    return !(std::fma(dx, vx, dy * vy) < kCutScaled);
}

}  // namespace

// log10_ratio: largest log10 of the covariance's eigenvalue ratio; centre_range:
// largest distance of the centre from the origin.  counts: Gaussians that are
// plain, boxes with an accepted pixel, boxes refused, accepted pixels in refused
// boxes (of plain Gaussians, of the others).
extern "C" void cutoff_check(uint64_t seed, int64_t n, double log10_ratio, double centre_range,
                             int64_t counts[5]) {
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> u01(0.0, 1.0);
    std::fill(counts, counts + 5, 0);
    const double sc = kScaleS;
    for (int64_t i = 0; i < n; ++i) {
        const double big = std::pow(10.0, 5.0 * u01(rng) - 1.0);           // eigenvalue
        const double small = big * std::pow(10.0, -log10_ratio * u01(rng));
        const double t = u01(rng) < 0.3 ? 0.25 * M_PI : M_PI * u01(rng);   // 45 degrees often
        const double c = std::cos(t), s = std::sin(t);
        Trial g;
        g.a = big * c * c + small * s * s;
        g.d = big * s * s + small * c * c;
        g.b = (big - small) * c * s;
        g.xc = centre_range * (2.0 * u01(rng) - 1.0);
        g.yc = centre_range * (2.0 * u01(rng) - 1.0);
        const double det = g.a * g.d - g.b * g.b;
        if (!(det > 0.0)) continue;
        const double Fa = g.d / det, Fd = g.a / det, Fc = -g.b / det;
        const float sfxx = (float)(sc * Fa), sfyy = (float)(sc * Fd), sfxy = (float)(sc * Fc);
        const float xcen = (float)g.xc, ycen = (float)g.yc;
        const float xlo = (float)(g.xc - (double)xcen), ylo = (float)(g.yc - (double)ycen);
        const bool is_plain = plain(g.xc, g.yc, sc * Fa, sc * Fd, sc * Fc, 1.0);
        counts[0] += is_plain;
        // a box of 8 x 8 pixels (or one row) with a point near the cutoff ellipse
        // at one of its places, mostly an edge or a corner
        const double e = std::sqrt(36.0 * (0.9 + 0.2 * u01(rng)));
        const double w = 2.0 * M_PI * u01(rng);
        const double p = e * std::sqrt(big) * std::cos(w), q = e * std::sqrt(small) * std::sin(w);
        const double px = g.xc + p * c - q * s, py = g.yc + p * s + q * c;
        const int rows = u01(rng) < 0.5 ? 8 : 1;
        const double ix = std::floor(px) - (int)(8 * u01(rng));
        const double iy = std::floor(py) - (int)(rows * u01(rng));
        const float x0 = (float)ix, x1 = (float)(ix + 7), y0 = (float)iy,
                    y1 = (float)(iy + rows - 1);
        bool any = false;
        for (int k = 0; k < 2 * 8 * rows; ++k) {
            const int j = k / 2;
            any |= inside((float)(ix + j % 8), (float)(iy + j / 8), xcen, ycen, xlo, ylo,
                          k % 2, sfxx, sfyy, sfxy);
        }
        bool visited;
        if (is_plain) {
            visited = meets(x0 - 0.01f - xcen, x1 + 0.01f - xcen, y0 - 0.01f - ycen,
                            y1 + 0.01f - ycen, sfxx, sfyy, sfxy);
        } else {
            const double hx = 6.0 * std::sqrt(g.a) * 1.001 + 0.01;
            const double hy = 6.0 * std::sqrt(g.d) * 1.001 + 0.01;
            visited = !((float)(g.xc + hx) < x0 || (float)(g.xc - hx) > x1 ||
                        (float)(g.yc + hy) < y0 || (float)(g.yc - hy) > y1);
        }
        counts[1] += any;
        counts[2] += !visited;
        if (any && !visited) ++counts[is_plain ? 3 : 4];
    }
}

// What meets() and plain() say of one Gaussian and one box about it.
extern "C" int cutoff_one(double xc, double yc, double sfxx, double sfyy, double sfxy,
                          double ampA, float xlo, float xhi, float ylo, float yhi) {
    return (plain(xc, yc, sfxx, sfyy, sfxy, ampA) ? 1 : 0) |
           (meets(xlo, xhi, ylo, yhi, (float)sfxx, (float)sfyy, (float)sfxy) ? 2 : 0);
}
