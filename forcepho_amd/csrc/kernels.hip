// kernels.hip -- gfx950 kernels of the forcepho likelihood-and-gradient path.
//
//   convert_kernel      proposal -> image-plane Gaussians + Jacobians
//                       (forcepho/src/compute_gaussians_kernel.cu:45-127,
//                        forcepho/src/common_kernel.cc:175-240)
//   eval_kernel<K>      per-pixel mixture, residual, chi2 and the 7 gradient
//                       partials per source (common_kernel.cc:57-143,
//                       compute_gaussians_kernel.cu:262-301); one wave per
//                       tile of 64*K pixels, no float atomics; LDS holds only
//                       each wave's own records, slot masks and activity bits.
//   residual_kernel, gradient_kernel<K>
//                       the same in two launches, for small plans: one wave
//                       per 64-pixel slot, then per (tile, source)
//   reduce_kernel       fixed-order sum of tile partials (FP64 or FP32)
//                       (replaces the shared-memory Accumulator,
//                        compute_gaussians_kernel.cu:133-198)
//   theta_kernel        parameter vector -> source records (FP32 fpho_source
//                       and/or FP64 Source64), Sersic amplitudes from
//                       bicubic B-splines in FP64 (forcepho/sources.py:607-694)
//   stack_kernel        lnlike = -chi2/2 and stacked gradient
//                       (forcepho/model.py:331-332,370-387)
//   step_kernel         bounded transform, its gradient and a leapfrog update
//                       (forcepho/model.py:302-368,596-636)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cutoff.h"
#include "fpho_internal.h"
#include "kernels.h"

namespace fpho {

// ------------------------------------------------------------------ convert

// Build one image Gaussian in FP64: the source set-up of
// compute_gaussians_kernel.cu:76-124 and the convolution and Jacobian of
// GetGaussianAndJacobian (common_kernel.cc:175-240).  The per-Gaussian cost
// is negligible next to the pixel pass, so it runs in double and is rounded
// once into the FP32 record the pixel pass streams.
// Returns the FPHO_STATUS_* bits of what it met (0 for a valid Gaussian).
// Src is fpho_source (the FP32 proposal record) or Source64 (the same fields
// in FP64, from the parameter-vector path).
template <typename Src>
__device__ __forceinline__ uint32_t make_image_gaussian(const ExpDesc &e, const Src &src,
                                                        int s, int p, ImgGauss &g,
                                                        ImgGauss64 &g64) {
    using M = M22<double>;
    const float *Dp = e.D + 4 * s;
    const float *CWp = e.CW + 4 * s;
    const M D{Dp[0], Dp[1], Dp[2], Dp[3]};

    double sn, cs;
    sincos((double)src.pa, &sn, &cs);
    const double q = src.q;
    const M R{cs, -sn, sn, cs};
    const M dR{-sn, -cs, cs, -sn};
    const double iq = 1.0 / q;
    const M S{iq, 0.0, 0.0, q};
    const M dS{-iq * iq, 0.0, 0.0, 1.0};

    const M DR = mul(D, R);
    const M T = mul(DR, S);
    const M dT_dq = mul(DR, dS);
    const M dT_dpa = mul(mul(D, dR), S);

    // source centre in pixels: CW (ra - crval, dec - crval) + crpix
    const double s0 = (double)src.ra - (double)e.crval[2 * s + 0];
    const double s1 = (double)src.dec - (double)e.crval[2 * s + 1];
    const double xs = (double)CWp[0] * s0 + (double)CWp[1] * s1 + (double)e.crpix[2 * s + 0];
    const double ys = (double)CWp[2] * s0 + (double)CWp[3] * s1 + (double)e.crpix[2 * s + 1];

    const fpho_psf_gauss pg = e.psf[p];
    const int bin = pg.sersic_radius_bin;
    const double r2 = e.rad2[bin];

    // covariance = r2 T T^T + C_psf ; F = covariance^-1
    const M Tt = transpose(T);
    const M cov = add(scale(mul(T, Tt), r2), M{pg.Cxx, pg.Cxy, pg.Cxy, pg.Cyy});
    const M F = inverse(cov);
    const double detF = det(F);

    const double flux = src.fluxes[e.band];
    const double am = src.mixture_amplitudes[bin];
    const double tmp = (double)e.G * (double)pg.amp * sqrt(detF) * (0.5 / 3.14159265358979323846);
    const double amp = tmp * flux * am;
    const double xc = xs + (double)pg.xcen - (double)e.x0;   // relative to the origin
    const double yc = ys + (double)pg.ycen - (double)e.y0;

    // dSigma = r2 (T dT^T + dT T^T); dF = -F dSigma F
    const M dSq = scale(add(mul(T, transpose(dT_dq)), mul(dT_dq, Tt)), r2);
    const M dSp = scale(add(mul(T, transpose(dT_dpa)), mul(dT_dpa, Tt)), r2);
    const M dFq = scale(mul(F, mul(dSq, F)), -1.0);
    const M dFp = scale(mul(F, mul(dSp, F)), -1.0);

    // bounding box of the cutoff ellipse d^T F d <= 36: |dx| <= 6 sqrt(cov_xx),
    // widened (0.1% + 0.01 pix) so that no pair the FP32 test accepts is
    // outside it; skipping boxed-out tiles then changes no result bit.
    const double hx = 6.0 * sqrt(cov.a) * 1.001 + 0.01;
    const double hy = 6.0 * sqrt(cov.d) * 1.001 + 0.01;
    g.xlo = order_key((float)(xc - hx));
    g.xhi = order_key((float)(xc + hx));
    g.ylo = order_key((float)(yc - hy));
    g.yhi = order_key((float)(yc + hy));

    // value parameters in the scaled variables of the pixel pass
    const double sc = kScaleS, sc2 = sc * sc;
    g.xcen = (float)xc;
    g.ycen = (float)yc;
    g.sfxx = (float)(sc * F.a);
    g.sfyy = (float)(sc * F.d);
    g.sfxy = (float)(sc * F.c);
    g.hcs = (float)(sc2 * (24.0 - F.a - F.d));
    g.ampA = (float)(amp / (24.0 * sc2));
    // |C| = |ampA| gp h' <= |ampA| (|hcs| + s^2 tr(F) max_E E e^{-E/2}), since
    // |v'|^2 <= s^2 lambda_max(F) E and E e^{-E/2} <= 2/e; widened by 1%
    g.peak = (float)(1.01 * fabs(amp / (24.0 * sc2)) *
                     (fabs(sc2 * (24.0 - F.a - F.d)) + sc2 * (F.a + F.d) * 0.73575888234288467));

    // gradient epilogue constants: Jacobian of (A, F) with respect to the
    // source parameters folded with amp and the powers of s (derivation in
    // eval_tile)
    const double dA_dq = 0.5 * amp * trace(mul(cov, dFq));
    const double dA_dpa = 0.5 * amp * trace(mul(cov, dFp));
    const double c24 = 1.0 / (24.0 * sc2);
    g.cA_flux = (float)(tmp * am * c24);
    g.cA_q = (float)(dA_dq * c24);
    g.cA_pa = (float)(dA_dpa * c24);
    g.cA_n = (float)(tmp * flux * src.damplitude_dnsersic[bin] * c24);
    g.cA_rh = (float)(tmp * flux * src.damplitude_drh[bin] * c24);
    g.k_axx = (float)(-amp / (48.0 * sc2));
    g.k_axy = (float)(-amp / (24.0 * sc2));
    g.k_e = (float)(-amp / 24.0);
    g.k_u = (float)(amp / (12.0 * sc));
    g.k_x1 = (float)(amp / (24.0 * sc2 * sc));
    g.k_x2 = (float)(-amp / (12.0 * sc2));
    g.dFxx_dQ = (float)dFq.a;
    g.dFyy_dQ = (float)dFq.d;
    g.dFxy_dQ = (float)dFq.c;
    g.dFxx_dPA = (float)dFp.a;
    g.dFyy_dPA = (float)dFp.d;
    g.dFxy_dPA = (float)dFp.c;
    g.xcen_lo = (float)(xc - (double)g.xcen);
    g.ycen_lo = (float)(yc - (double)g.ycen);
    g.pad1 = 0.0f;

    g64.xcen = xc;
    g64.ycen = yc;
    g64.sfxx = sc * F.a;
    g64.sfyy = sc * F.d;
    g64.sfxy = sc * F.c;
    g64.hcs = sc2 * (24.0 - F.a - F.d);
    g64.ampA = amp / (24.0 * sc2);
    g64.pad0 = 0.0;

    // what the reference would turn into NaN or Inf silently
    uint32_t flags = 0;
    if (!(isfinite(src.ra) && isfinite(src.dec) && isfinite(src.q) && isfinite(src.pa) &&
          isfinite(flux) && isfinite(am) && isfinite(src.damplitude_dnsersic[bin]) &&
          isfinite(src.damplitude_drh[bin])))
        flags |= FPHO_STATUS_PROPOSAL_NONFINITE;
    if (!(src.q > 0)) flags |= FPHO_STATUS_Q_NONPOSITIVE;
    if (!(det(cov) > 0.0)) flags |= FPHO_STATUS_COVARIANCE;
    if (!(isfinite(amp) && isfinite(xc) && isfinite(yc) && isfinite(F.a) && isfinite(F.c) &&
          isfinite(F.d) && isfinite(dA_dq) && isfinite(dA_dpa)))
        flags |= FPHO_STATUS_GAUSSIAN_NONFINITE;
    return flags;
}

// Workgroups (exposure, part): one wave each, its lanes stride over the
// exposure's n_src * n_psf Gaussians in steps of gridDim.y waves.  Bound by the
// latency of one Gaussian's FP64 chain (sincos, divisions, square roots), so
// the Gaussians are spread until the chip holds a wave or two per SIMD; one
// workgroup of 128 lanes per exposure ran a chain per 128 Gaussians (us, before
// -> after: four patches of up to 1620 Gaussians an exposure 20.7 -> 9.8, 24
// exposures of 2160 46.6 -> 9.4, 96 patches 116 -> 106).
// Invalid inputs set bits of *status (a vector atomic, taken only then).
template <typename Src>
__global__ __launch_bounds__(kWave) void convert_kernel(
    const ExpDesc *__restrict__ exps, const Src *__restrict__ props,
    ImgGauss *__restrict__ out, ImgGauss64 *__restrict__ out64, int4 *__restrict__ boxes,
    HotGauss *__restrict__ hot, uint32_t *__restrict__ status) {
    const ExpDesc &e = exps[blockIdx.x];
    const int n = e.n_src * e.n_psf;
    for (int j = blockIdx.y * kWave + threadIdx.x; j < n; j += gridDim.y * kWave) {
        const int s = j / e.n_psf;
        const int p = j - s * e.n_psf;
        ImgGauss g;
        ImgGauss64 g64;
        const uint32_t flags = make_image_gaussian(e, props[e.src_off + s], s, p, g, g64);
        if (flags) atomicOr(status, flags);
        out[e.gauss_off + j] = g;
        out64[e.gauss_off + j] = g64;
        boxes[e.gauss_off + j] = make_int4(g.xlo, g.xhi, g.ylo, g.yhi);
        if (hot)
            hot[e.gauss_off + j] = {g.xcen, g.ycen, g.sfxx, g.sfyy, g.sfxy, g.hcs, g.ampA,
                                    plain(g64.xcen, g64.ycen, g64.sfxx, g64.sfyy, g64.sfxy, g64.ampA)
                                        ? 0u
                                        : kNotPlain};
    }
}

// --------------------------------------------------------------- pixel pass

constexpr float kMaskedCoord = 1.0e6f;  // lanes past the tile end: far away

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// True when the Gaussian's cutoff box (gb = xlo, xhi, ylo, yhi keys) misses
// the tile's pixel box tb; integer compares only.
__device__ __forceinline__ bool boxed_out(int cull, const int4 gb, const int4 tb) {
    const int miss = (gb.y < tb.x ? 1 : 0) | (gb.x > tb.y ? 2 : 0) | (gb.w < tb.z ? 4 : 0) |
                     (gb.z > tb.w ? 8 : 0);
    return cull != 0 && miss != 0;
}

// Value of one image Gaussian at one pixel in FP64 (bright terms only), in
// the scaled variables of ImgGauss: ampA 2^E' (hcs + v'.v').  2^E' for
// E' in [36 s, 0] is 2^n 2^f with n = rint(E'), |f| <= 1/2, and 2^f =
// (e^y)^1024 with y = f ln2 / 1024, |y| < 3.4e-4, e^y by its cubic Taylor
// polynomial (truncation 6e-16, amplified 1024-fold by the squarings to
// < 1e-12 relative) -- two constants, so the rare FP64 path holds few
// registers.
// Returns r - value (the subtraction fused with the last product).  The fused
// forms are written out, here and in the pair functions below, so that every
// kernel that evaluates a pair rounds it the same way.
__device__ __forceinline__ double minus_value64(double r, const ImgGauss64 &g, float xp, float yp) {
    const double dx = (double)xp - g.xcen;
    const double dy = (double)yp - g.ycen;
    const double vx = fma(g.sfxx, dx, g.sfxy * dy);
    const double vy = fma(g.sfxy, dx, g.sfyy * dy);
    const double ea = fma(dx, vx, dy * vy);
    const double n = __builtin_rint(ea);
    const double y = (ea - n) * (0.69314718055994530942 / 1024.0);
    double p = fma(y, fma(y, fma(y, 1.0 / 6.0, 0.5), 1.0), 1.0);
#pragma unroll
    for (int j = 0; j < 10; ++j) p *= p;
    const double h = fma(vx, vx, fma(vy, vy, g.hcs));
    return fma(-h, g.ampA * __builtin_ldexp(p, (int)n), r);
}

// Pass 1 of one pair: v' and the scaled exponent E' = s E.
__device__ __forceinline__ float exponent1(float dx, float dy, float sfxx, float sfyy, float sfxy,
                                           float &vx, float &vy) {
    vx = fmaf(sfxx, dx, sfxy * dy);
    vy = fmaf(sfyy, dy, sfxy * dx);
    return fmaf(dx, vx, dy * vy);
}

// exp2(E') of a pair; a pair beyond the cutoff gives an exact zero.
__device__ __forceinline__ float cut_exp(bool in, float ea) {
    return __builtin_amdgcn_exp2f(in ? ea : -__builtin_huge_valf());
}

// c2 + (r^2 - d^2) ierr^2 of one pixel; rd holds an FP32 residual when the
// residual is not kept in FP64.
template <bool MIXED>
__device__ __forceinline__ double add_chi2(double c2, double rd, float d, float ierr) {
    if (MIXED) {
        const double ie = (double)ierr, ds = (double)d * ie;
        return fma(fma(rd, ie, -ds), fma(rd, ie, ds), c2);
    }
    const float rs = (float)rd * ierr;
    const float ds = d * ierr;
    return fma((double)rs - (double)ds, (double)rs + (double)ds, c2);
}

// The 12 pixel sums of one Gaussian that its derivatives are linear in.
struct GradSums {
    float PA = 0.f, X1 = 0.f, X2 = 0.f, Y1 = 0.f, Y2 = 0.f, Pxx = 0.f;
    float Pyy = 0.f, Pxy = 0.f, Pe = 0.f, Peu = 0.f, Pea = 0.f, Pecr = 0.f;

    // one pixel at offset (dx, dy) with rr = -2 r ierr^2
    __device__ __forceinline__ void add(float dx, float dy, float rr, float sfxx, float sfyy,
                                        float sfxy, float hcs) {
        const float vx = fmaf(sfxx, dx, sfxy * dy);
        const float vy = fmaf(sfyy, dy, sfxy * dx);
        const float u = dx * vx;
        const float ea = fmaf(dy, vy, u);
        // a pixel beyond the cutoff gets gp = exp2(-inf) = 0, so all its
        // terms below are exact zeros (every factor is finite)
        const float gp = cut_exp(!(ea < kCutScaled), ea);
        const float h = fmaf(vx, vx, fmaf(vy, vy, hcs));
        const float ee = rr * gp;
        const float a = ee * h;
        PA = fmaf(ee, h, PA);
        X1 = fmaf(a, vx, X1);
        X2 = fmaf(ee, vx, X2);   // sum e v'x (s F applied in partials)
        Y1 = fmaf(a, vy, Y1);
        Y2 = fmaf(ee, vy, Y2);   // sum e v'y
        const float ax = a * dx;
        const float ay = a * dy;
        Pxx = fmaf(ax, dx, Pxx);
        Pxy = fmaf(ax, dy, Pxy);
        Pyy = fmaf(ay, dy, Pyy);
        Pe = fmaf(rr, gp, Pe);
        Peu = fmaf(ee, u, Peu);
        Pea = fmaf(ee, ea, Pea);
        Pecr = fmaf(ee, fmaf(dy, vx, dx * vy), Pecr);
    }
};

// v + the value OFF lanes on, in rows of 16 lanes.
template <int OFF>
__device__ __forceinline__ float add_ror(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 | OFF, 0xf,
                                                          0xf, true));
}

// Lanes 0-31: a + the value of a 32 lanes on; lanes 32-63: the same of b.
__device__ __forceinline__ float add_halves(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                    false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Rows 0 and 2: a + the value of a 16 lanes on; rows 1 and 3: the same of b.
__device__ __forceinline__ float add_rows(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
                                                    false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Row r (of 16 lanes) of the result holds the wave's sum of v_r, its additions
// paired as a butterfly's over lanes 32, 16, 8, 4, 2, 1 apart.  Four sums share
// the first two steps' additions and the lanes move in registers: a source's
// seven sums took 42 LDS shuffles (90 exposures, 13 sources: 955 -> 932 us a
// pass).
__device__ __forceinline__ float wave_sum4(float v0, float v1, float v2, float v3) {
    float v = add_rows(add_halves(v0, v2), add_halves(v1, v3));
    v = add_ror<8>(v);
    v = add_ror<4>(v);
    v = add_ror<2>(v);
    return add_ror<1>(v);
}

// A source's 7 partials over the pixels of one lane (position in pixels).
struct SourcePartials {
    float p0 = 0.f, sx = 0.f, sy = 0.f, p3 = 0.f, p4 = 0.f, p5 = 0.f, p6 = 0.f;

    // per-Gaussian epilogue: image-space derivative sums -> 7 partials
    __device__ __forceinline__ void add(const ImgGauss &G, float sfxx, float sfyy, float sfxy,
                                        const GradSums &q) {
        const float ke = G.k_e * q.Pe;
        const float gfx = fmaf(G.k_u, q.Peu, fmaf(G.k_axx, q.Pxx, ke));
        const float gfy = fmaf(G.k_u, q.Pea - q.Peu, fmaf(G.k_axx, q.Pyy, ke));
        const float gfxy = fmaf(G.k_u, q.Pecr, G.k_axy * q.Pxy);
        p0 = fmaf(G.cA_flux, q.PA, p0);
        p5 = fmaf(G.cA_n, q.PA, p5);
        p6 = fmaf(G.cA_rh, q.PA, p6);
        p3 = fmaf(G.cA_q, q.PA, p3);
        p3 = fmaf(G.dFxx_dQ, gfx, p3);
        p3 = fmaf(G.dFyy_dQ, gfy, p3);
        p3 = fmaf(G.dFxy_dQ, gfxy, p3);
        p4 = fmaf(G.cA_pa, q.PA, p4);
        p4 = fmaf(G.dFxx_dPA, gfx, p4);
        p4 = fmaf(G.dFyy_dPA, gfy, p4);
        p4 = fmaf(G.dFxy_dPA, gfxy, p4);
        // sum e (sF v')_x = sfxx sum e v'x + sfxy sum e v'y (and for y)
        const float fX = fmaf(sfxx, q.X2, sfxy * q.Y2);
        const float fY = fmaf(sfxy, q.X2, sfyy * q.Y2);
        sx = fmaf(G.k_x1, q.X1, fmaf(G.k_x2, fX, sx));
        sy = fmaf(G.k_x1, q.Y1, fmaf(G.k_x2, fY, sy));
    }

    // sum over the wave and write; the sky-position derivatives share the
    // source's CW matrix
    __device__ __forceinline__ void write(float *__restrict__ o, const float *__restrict__ CW,
                                          int lane) {
        const float u = wave_sum4(sx, p0, p3, p4), v = wave_sum4(sy, p5, p6, 0.0f);
        if ((lane & 15) == 0) {
            const int row = lane >> 4;
            const float dra = fmaf(CW[0], u, CW[2] * v);   // dx/dalpha, dy/dalpha
            const float ddec = fmaf(CW[1], u, CW[3] * v);  // dx/ddelta, dy/ddelta
            o[row == 0 ? 1 : row == 1 ? 0 : row + 1] = row == 0 ? dra : u;
            if (row < 3) o[row == 0 ? 2 : row + 4] = row == 0 ? ddec : v;
        }
    }
};

// A pointer known to be to device memory (descriptors hold generic ones), so
// loads take a scalar base and a 32-bit lane offset.
template <typename T>
using Global = const T __attribute__((address_space(1))) *;
template <typename T>
__device__ __forceinline__ Global<T> global(const T *p) {
    return (Global<T>)p;
}

// Set bits of m below this lane.
__device__ __forceinline__ int rank_in(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// LDS written by lanes of this wave is visible to its other lanes.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The value parameters of Gaussian i; tag: the bits of its peak.
__device__ __forceinline__ HotGauss load_record(const ImgGauss *__restrict__ g, uint32_t i) {
    const Global<float4> p = global(reinterpret_cast<const float4 *>(g)) +
                             sizeof(ImgGauss) / 16 * i + 1;
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 1);
    return {a.x, a.y, a.z, a.w, b.x, b.y, b.z, __float_as_uint(b.w)};
}

// Evaluate one wave tile.  `tile` must be wave-uniform (an SGPR value) so
// every descriptor load below is a scalar load.  Bound by VALU issue: an FMA
// with a scalar operand issues every 4.1 cycles here, one whose operands are
// all vector registers every 3.0, so both passes take the value
// parameters of the Gaussians they visit from LDS (64 are put there at once,
// a visit reads its own with a broadcast) and only the epilogue's constants by
// scalar loads.  Against scalar loads throughout: 96 patches of 228564 tiles,
// K = 8, 12440 -> 11730 us (0.35 -> 0.38 VALU instructions a cycle and SIMD);
// 530123 tiles, K = 4, 19470 -> 17260.
//   MIXED = true : residual accumulated in FP64; a term whose FP32 value
//                  exceeds kBrightSigma * sigma of the tile's quietest pixel
//                  is re-evaluated in FP64 (a wave branch taken only near
//                  bright cores; about 3% of slot evaluations on 512 uneven
//                  patches of 32^2-256^2 pixel exposures).
//   MIXED = false: FP32 residual, as forcepho/src/common_kernel.cc:57-83.
//
// Scaled variables (ImgGauss): d = pixel - centre, v' = s F d, E' = d.v' =
// s E, gp = exp(-E/2) = exp2(E'), h' = hcs + v'.v' = 24 s^2 H.
// Gradient (common_kernel.cc:95-143): with e = -2 r ierr^2 gp and
// a = e H = a' / (24 s^2), a' = e h', the reference's per-pair terms are
//   dC/dA   = a
//   dC/dx   = amp (a vx - e (F v)_x / 12)
//   dC/dFxx = amp (-a dx^2 / 2 - e / 24 + e dx vx / 12)
//   dC/dFyy = amp (-a dy^2 / 2 - e / 24 + e dy vy / 12)
//   dC/dFxy = amp (-a dx dy + e (dy vx + dx vy) / 12)
// With v = v'/s, F v = (s F v')/s^2, dx vx = u'/s (u' = dx v'x), they are
// linear in 12 pixel sums of a', a' v'x, e v'x, a' v'y, e v'y,
// a' dx^2, a' dy^2, a' dx dy, e, e u', e w' (w' = dy v'y), e cr'
// (cr' = dy v'x + dx v'y); each sum costs one FMA per pair (e w' is kept as
// e E' = e (u' + w') and e u' subtracted once) and is turned into the 7
// source partials once per Gaussian (constants in ImgGauss).
//
// Pass 1 tests the cutoff boxes of 64 Gaussians at once (one vector load, a
// ballot) against the boxes of the tile's 64-pixel slots and visits, in
// index order, only those that meet a slot, at those slots.  It
// records, per Gaussian, which of the K pixel slots hold a pixel inside the
// cutoff (a K-bit mask, one byte in LDS per Gaussian for the first mask_cap
// Gaussians) and which Gaussians have any (one bit each in LDS, 64 per word,
// for the first 64 act_words Gaussians); pass 2 visits only those Gaussians
// and evaluates only those slots.  Gaussians past either capacity are
// visited with every slot: a pixel beyond the cutoff adds exact zeros.
template <int K, bool MIXED, bool CENTRE>
__device__ __forceinline__ void eval_tile(int tile, const TileDesc *__restrict__ tiles,
                                          const ExpDesc *__restrict__ exps,
                                          const ImgGauss *__restrict__ gauss,
                                          const ImgGauss64 *__restrict__ gauss64,
                                          const int4 *__restrict__ gboxes,
                                          const int4 *__restrict__ slot_boxes,
                                          float *__restrict__ gpart,
                                          double *__restrict__ cpart, int cull,
                                          uint8_t *__restrict__ amask, int mask_cap,
                                          uint64_t *__restrict__ act, int act_words,
                                          HotGauss *__restrict__ rec) {
    const int lane = threadIdx.x & (kWave - 1);
    const TileDesc t = tiles[tile];
    const ExpDesc &e = exps[t.exp];
    const ImgGauss *__restrict__ g = gauss + e.gauss_off;
    const ImgGauss64 *__restrict__ g64 = gauss64 + e.gauss_off;
    const int4 *__restrict__ gb = gboxes + e.gauss_off;
    const int n_src = e.n_src;
    const int n_psf = e.n_psf;
    const int ng = n_src * n_psf;

    float x[K], y[K], r[K];
    double rd[K];
    float tmin = __builtin_huge_valf();   // smallest bright threshold in the tile
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int p = k * kWave + lane;
        float dk = 0.0f;
        if (p < t.npix) {
            const int i = t.pix0 + p;
            x[k] = e.xpix[i] - e.x0;
            y[k] = e.ypix[i] - e.y0;
            dk = e.data[i];
            const float iek = e.ierr[i];
            if (MIXED && iek > 0.0f) tmin = fminf(tmin, kBrightSigma / iek);
        } else {
            x[k] = kMaskedCoord;
            y[k] = kMaskedCoord;
        }
        r[k] = dk;
        rd[k] = (double)dk;
    }

    // A Gaussian whose cutoff box misses the box of a 64-pixel slot adds
    // nothing to that slot's pixels.  Lane k < K holds slot k's box; a slot
    // with no pixel has an empty box.
    int4 sbox = make_int4(INT_MAX, INT_MIN, INT_MAX, INT_MIN);
    if (lane < K && lane * kWave < t.npix) sbox = slot_boxes[t.chunk0 + lane];

    // A term counts as bright above 0.1 sigma of the tile's quietest pixel;
    // a Gaussian whose peak stays below that cannot have a bright term here.
    if (MIXED) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) tmin = fminf(tmin, __shfl_xor(tmin, off, kWave));
        // readfirstlane is an integer builtin: pass the float's bits
        tmin = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tmin)));
    }

    // ---- pass 1: residual = data - sum_g C_g   (common_kernel.cc:57-83)
    // The boxes of 64 Gaussians are tested at once (lane j: Gaussian
    // base + j) against the K slot boxes; only Gaussians whose box meets a
    // slot are visited, in order, and only at those slots.  act[] keeps, per
    // 64 Gaussians, the ones with a pixel inside the cutoff.
    for (int base = 0; base < ng; base += kWave) {
        const int j = base + lane;
        uint32_t sm = 0;   // slots whose box meets Gaussian j's box
        if (j < ng) {
            if (cull) {
                const int4 b = gb[j];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int4 q = make_int4(__builtin_amdgcn_readlane(sbox.x, k),
                                             __builtin_amdgcn_readlane(sbox.y, k),
                                             __builtin_amdgcn_readlane(sbox.z, k),
                                             __builtin_amdgcn_readlane(sbox.w, k));
                    sm |= boxed_out(1, b, q) ? 0u : 1u << k;
                }
            } else {
                sm = (1u << K) - 1;
            }
        }
        const uint64_t todo = __builtin_amdgcn_ballot_w64(sm != 0);
        const int cnt = __builtin_popcountll(todo);
        if (sm != 0) {
            HotGauss h = load_record(g, (uint32_t)j);
            // h.tag: the peak's bits
            const bool bright = __uint_as_float(h.tag) > tmin;
            h.tag = (MIXED && bright ? 1u << 31 : 0u) | (uint32_t)lane << 8 | sm;
            rec[rank_in(todo)] = h;
        }
        wave_lds_sync();
        uint64_t active = 0;
        for (int n = 0; n < cnt; ++n) {
            const HotGauss H = rec[n];
            const uint32_t tag = __builtin_amdgcn_readfirstlane(H.tag);
            const int bit = (tag >> 8) & 63;
            const int i = base + bit;
            uint32_t m = 0;   // slots with a pixel inside the cutoff (wave-uniform)
            const float xcl = CENTRE ? g[i].xcen_lo : 0.0f, ycl = CENTRE ? g[i].ycen_lo : 0.0f;
            // a term is bright when |c| > tb: a Gaussian whose peak stays
            // below the tile threshold cannot have one
            const float tb = tag >> 31 ? tmin : __builtin_huge_valf();
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (!(tag & (1u << k))) continue;
                float dx = x[k] - H.xcen;
                float dy = y[k] - H.ycen;
                if (CENTRE) {   // the pixel offset from the FP64 centre
                    dx -= xcl;
                    dy -= ycl;
                }
                float vx, vy;
                const float ea = exponent1(dx, dy, H.sfxx, H.sfyy, H.sfxy, vx, vy);   // s E
                const bool in = !(ea < kCutScaled);       // E <= 36 (cutoff)
                if (__builtin_amdgcn_ballot_w64(in) == 0) continue;
                m |= 1u << k;
                {
                    // a lane beyond the cutoff adds an exact zero
                    const float gp = cut_exp(in, ea);
                    const float h = fmaf(vx, vx, fmaf(vy, vy, H.hcs));
                    const float c = H.ampA * gp * h;
                    if (MIXED) {
                        if (fabsf(c) > tb) {
                            // keep the FP64 copies of the coordinates inside
                            // this rare branch (hoisted out of the Gaussian
                            // loop they would hold 4K more registers)
                            float xk = x[k], yk = y[k];
                            asm volatile("" : "+v"(xk), "+v"(yk));
                            rd[k] = minus_value64(rd[k], g64[i], xk, yk);
                        } else
                            rd[k] -= (double)c;
                    } else {
                        r[k] -= c;
                    }
                }
            }
            if (m) active |= 1ull << bit;
            if (i < mask_cap && lane == 0) amask[i] = (uint8_t)m;
        }
        if (lane == 0 && base / kWave < act_words) act[base / kWave] = active;
        wave_lds_sync();   // before the next 64 Gaussians' records
    }

    // pass 2 of this wave reads the masks and activity words of its lane 0
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // ---- chi2 = sum (r^2 - d^2) ierr^2 in FP64 (compute_gaussians_kernel.cu:276-287)
    // (pixel indices recomputed from an opaque copy of the lane id: kept
    // from the load above, they would hold K registers across pass 1)
    int lane2 = lane;
    asm volatile("" : "+v"(lane2));
    double c2 = 0.0;
    float rr[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int p = k * kWave + lane2;
        float dk = 0.0f, iek = 0.0f;
        if (p < t.npix) {
            dk = e.data[t.pix0 + p];
            iek = e.ierr[t.pix0 + p];
        }
        if (MIXED) r[k] = (float)rd[k];
        c2 = add_chi2<MIXED>(c2, MIXED ? rd[k] : (double)r[k], dk, iek);
        if (e.residual != nullptr && p < t.npix) e.residual[t.pix0 + p] = r[k];
        rr[k] = -2.0f * ((r[k] * iek) * iek);  // -2 r ierr^2
        // finish this slot here: deferred, its loaded values would spill
        asm volatile("" : "+v"(c2), "+v"(rr[k]));
    }
    c2 = wave_sum(c2);
    if (lane == 0) cpart[tile] = c2;

    // ---- pass 2: per source, 7 partials   (common_kernel.cc:95-143)
    float *__restrict__ out = gpart + t.part_off;
    for (int s = 0; s < n_src; ++s) {
        SourcePartials src;
        const int i0 = s * n_psf;
        bool touched = false;
        for (int cb = 0; cb < n_psf; cb += kWave) {
            // lane l: Gaussian i and the slots to evaluate: pass 1's mask, else
            // (past the LDS capacity) every slot
            const bool valid = cb + lane < n_psf;
            const int i = i0 + (valid ? cb + lane : 0);
            const int w = i / kWave;
            const uint64_t word = w < act_words ? act[w] : ~0ull;
            const bool in = valid && ((word >> (i & (kWave - 1))) & 1);
            const uint64_t hits = __builtin_amdgcn_ballot_w64(in);
            const int cnt = __builtin_popcountll(hits);
            if (cnt == 0) continue;
            touched = true;
            if (in) {
                HotGauss h = load_record(g, (uint32_t)i);
                h.tag = (uint32_t)i << 8 | (i < mask_cap ? amask[i] : 0xFFu);
                rec[rank_in(hits)] = h;
            }
            wave_lds_sync();
            for (int n = 0; n < cnt; ++n) {
                const HotGauss H = rec[n];
                const uint32_t v = __builtin_amdgcn_readfirstlane(H.tag);
                const ImgGauss &G = g[v >> 8];
                const float xcl = CENTRE ? G.xcen_lo : 0.0f, ycl = CENTRE ? G.ycen_lo : 0.0f;
                GradSums q;   // over this lane's K pixels
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    if (!(v & (1u << k))) continue;
                    float dx = x[k] - H.xcen;
                    float dy = y[k] - H.ycen;
                    if (CENTRE) {
                        dx -= xcl;
                        dy -= ycl;
                    }
                    q.add(dx, dy, rr[k], H.sfxx, H.sfyy, H.sfxy, H.hcs);
                }
                src.add(G, H.sfxx, H.sfyy, H.sfxy, q);
            }
            wave_lds_sync();   // before the next 64 Gaussians' records
        }
        float *o = out + kNParams * s;
        if (!touched) {
            // no Gaussian of this source reaches the tile
            if (lane < kNParams) o[lane] = 0.0f;
            continue;
        }
        src.write(o, e.CW + 4 * s, lane);
    }
}

// Workgroup b runs on XCD b % 8 (round-robin dispatch); map it to queue
// group (chunk-row, XCD, offset) so that each XCD takes chunks of C
// consecutive groups (tiles of one exposure share image Gaussians in its L2
// and scalar caches) and the chunks interleave across XCDs (the cost-sorted
// queue stays balanced).  A bijection on [0, n); the tail past the last full
// row of 8*C groups maps to itself.
constexpr int kXcdChunk = 64;   // queue groups per XCD chunk (measured: 16, 64, 256)

template <int C>
__device__ __forceinline__ int xcd_swizzle(int b, int n) {
    constexpr int X = 8, span = X * C;
    const int full = (n / span) * span;
    if (b >= full) return b;
    const int xcd = b % X, local = b / X;
    return (local / C) * span + xcd * C + (local % C);
}

// Eight waves per SIMD (the most a SIMD holds) caps the kernels at 64
// VGPRs (measured at K = 8: 5.7% faster than 6 waves at 76 VGPRs); the kernels
// that keep a tile's residuals spill a few values once per tile.
#define FPHO_EVAL_OCCUPANCY __attribute__((amdgpu_waves_per_eu(8)))

// Non-persistent: wave w of workgroup b evaluates queue[b*W + w].
template <int K, bool MIXED, bool CENTRE>
__global__ __launch_bounds__(256) FPHO_EVAL_OCCUPANCY void eval_kernel(
    const TileDesc *__restrict__ tiles, const int32_t *__restrict__ queue,
    int32_t n_tiles, int32_t waves_per_group, const ExpDesc *__restrict__ exps,
    const ImgGauss *__restrict__ gauss, const ImgGauss64 *__restrict__ gauss64,
    const int4 *__restrict__ gboxes, const int4 *__restrict__ slot_boxes,
    float *__restrict__ gpart, double *__restrict__ cpart,
    int32_t cull, int32_t mask_cap, int32_t act_words) {
    extern __shared__ HotGauss lds_records[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = xcd_swizzle<kXcdChunk>((int)blockIdx.x, (int)gridDim.x) *
                     waves_per_group + w;
    if (slot >= n_tiles) return;
    const int tile = __builtin_amdgcn_readfirstlane(queue[slot]);
    uint8_t *lds_mask = reinterpret_cast<uint8_t *>(lds_records + waves_per_group * kWave);
    eval_tile<K, MIXED, CENTRE>(tile, tiles, exps, gauss, gauss64, gboxes, slot_boxes, gpart, cpart,
                        cull, lds_mask + w * mask_cap, mask_cap,
                        reinterpret_cast<uint64_t *>(lds_mask + waves_per_group * mask_cap) +
                            w * act_words, act_words, lds_records + w * kWave);
}

// Persistent: every wave pulls tiles from `counter` until the queue is empty.
// Each wave reaches the exit once the counter passes n_tiles.
template <int K, bool MIXED, bool CENTRE>
__global__ __launch_bounds__(256) FPHO_EVAL_OCCUPANCY void eval_persistent_kernel(
    const TileDesc *__restrict__ tiles, const int32_t *__restrict__ queue,
    int32_t n_tiles, int32_t *__restrict__ counter, const ExpDesc *__restrict__ exps,
    const ImgGauss *__restrict__ gauss, const ImgGauss64 *__restrict__ gauss64,
    const int4 *__restrict__ gboxes, const int4 *__restrict__ slot_boxes,
    float *__restrict__ gpart, double *__restrict__ cpart,
    int32_t cull, int32_t mask_cap, int32_t act_words) {
    extern __shared__ HotGauss lds_records[];
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = (int)(blockDim.x >> 6);
    uint8_t *lds_mask = reinterpret_cast<uint8_t *>(lds_records + W * kWave);
    for (;;) {
        int slot = 0;
        if (lane == 0) slot = atomicAdd(counter, 1);
        slot = __builtin_amdgcn_readfirstlane(__shfl(slot, 0, kWave));
        if (slot >= n_tiles) break;
        const int tile = __builtin_amdgcn_readfirstlane(queue[slot]);
        eval_tile<K, MIXED, CENTRE>(tile, tiles, exps, gauss, gauss64, gboxes, slot_boxes, gpart,
                            cpart, cull, lds_mask + w * mask_cap, mask_cap,
                            reinterpret_cast<uint64_t *>(lds_mask + W * mask_cap) +
                                w * act_words, act_words, lds_records + w * kWave);
    }
}

// ------------------------------------------------ pixel pass in two launches
//
// For plans whose tiles do not fill the chip many times over, with exposures not
// much wider than a source reaches (two_launches() in runtime.hip):
// residual_kernel runs one wave per 64-pixel slot, gradient_kernel one wave
// per (tile, source), so a tile's work is spread over its slots and then over
// its sources instead of being one wave's.  A pixel's Gaussians are still
// subtracted in index order by one lane, a source's partials are still summed
// over the tile's K slots by one wave, and pass 2 visits the slots that pass
// 1 found active, so every result is eval_tile's bit for bit.
//
// What bounds it: VALU issue, and on small plans the serial chain of the
// heaviest wave.  Measured (us, one wave per tile -> two launches): 16 tiles
// of 54 Gaussians 58 -> 26; 2048 tiles of 720 535 -> 216; 6144 tiles of 2160
// 1440 -> 895; 611 tiles of up to 1620 (four patches) 882 -> 126.

// xcd_swizzle with the XCDs' chunks moved on from row to row: an exposure is
// often a whole number of chunks, and without that an XCD would take the same
// part of every exposure, its crowded middle or its empty edge.  Any odd step
// meets all 8 XCDs; by three, 60 sources on 24 exposures of 256^2 take 947 us a
// pass (1013 without), 13 on 90 of 256^2 942 (972).
// turn: how far a chunk's waves turn from row to row as well.  Waves are dealt to
// the CUs in order, so without it the same CU takes the same place of every
// exposure.  29 is odd, so that it meets all places of a chunk, and near half
// of 64: in the residual launch 20 sources on 32 exposures of 128^2 take 240 us
// (248 without), the 60 sources 947 (932); the gradient launch goes source by
// source and loses 1% by it.
// Chunks of 128 waves from 2^15 waves on, else of 64 (90 exposures 942 us, all 64
// 951, all 128 954).  Exposures that are no whole number of chunks (97^2) gain or
// lose under 4% by any of the three.
__device__ __forceinline__ int xcd_rotate(int b, int n, int turn) {
    const int shift = n >= 1 << 15 ? 7 : 6;   // log2 of the chunk
    const int rows = n >> (shift + 3);
    if (b >= rows << (shift + 3)) return b;
    const int local = b >> 3, row = local >> shift;
    const int xcd = (b + 3 * row) & 7;
    return (((row << 3) + xcd) << shift) + ((local + turn * row) & ((1 << shift) - 1));
}

// The record of Gaussian i (two 16-byte loads).
__device__ __forceinline__ HotGauss load_hot(const HotGauss *__restrict__ hot, uint32_t i) {
    const Global<float4> p = global(reinterpret_cast<const float4 *>(hot)) + 2 * i;
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 1);
    return {a.x, a.y, a.z, a.w, b.x, b.y, b.z, __float_as_uint(b.w)};
}

// Pass 1 of one slot.  Each block of 64 Gaussians is tested at once (lane j:
// Gaussian base + j) and the records of those that meet the slot go to LDS in
// index order, from where a visit reads its own with a broadcast.  An FMA
// with a scalar operand issues every 4.1 cycles here, one whose operands are
// all vector registers every 3.0; 8 of a visit's 18 instructions read the
// record, so taking it from LDS instead of by scalar loads cut the kernel from
// 460 to 360 us (24576 slots, 2160 Gaussians) and from 142 to 120 (8192, 720).
// kVisits go through together: one wait for their records and one test for
// bright terms (four small patches: 218 us a pass with four, 232 with two).
// A block that holds a Gaussian that is not plain() goes one visit at a time,
// as eval_tile does: such a Gaussian is tested by its cutoff box, is visited
// only where a lane is inside its cutoff, and is bright only above its peak.
template <int K, bool MIXED, bool CENTRE>
__global__ __launch_bounds__(kWave) FPHO_EVAL_OCCUPANCY void residual_kernel(
    const TileDesc *__restrict__ tiles, const int32_t *__restrict__ queue,
    const ExpDesc *__restrict__ exps, const ImgGauss *__restrict__ gauss,
    const ImgGauss64 *__restrict__ gauss64, const HotGauss *__restrict__ hot,
    const int4 *__restrict__ gboxes, const int4 *__restrict__ slot_boxes,
    uint64_t *__restrict__ flags, double *__restrict__ resid, float *__restrict__ weight,
    int32_t cull) {
    constexpr int kVisits = 4;
    const int lane = threadIdx.x;
    const int wave = xcd_rotate((int)blockIdx.x, (int)gridDim.x, 29);
    const TileDesc t = tiles[queue[wave / K]];
    const int k = wave % K;
    const int npix = t.npix - k * kWave;   // of this slot and the ones after it
    if (npix <= 0) return;
    const int pix0 = t.pix0 + k * kWave;
    const ExpDesc &e = exps[t.exp];
    const int4 box = slot_boxes[t.chunk0 + k];
    // 0.01 pixel covers the FP32 rounding of the centre
    const float xlo = key_float(box.x) - 0.01f, xhi = key_float(box.y) + 0.01f;
    const float ylo = key_float(box.z) - 0.01f, yhi = key_float(box.w) + 0.01f;
    // no Gaussian counts as plain on a slot beyond the coordinates of plain()
    const uint64_t far = __builtin_amdgcn_ballot_w64(
        !(fmaxf(fmaxf(-xlo, xhi), fmaxf(-ylo, yhi)) < kMaskedCoord));
    const ImgGauss *__restrict__ g = gauss + e.gauss_off;
    const ImgGauss64 *__restrict__ g64 = gauss64 + e.gauss_off;
    const int ng = e.n_src * e.n_psf;

    float x = kMaskedCoord, y = kMaskedCoord, r = 0.0f, iek = 0.0f;
    if (lane < npix) {
        x = global(e.xpix + pix0)[(uint32_t)lane] - e.x0;
        y = global(e.ypix + pix0)[(uint32_t)lane] - e.y0;
        r = global(e.data + pix0)[(uint32_t)lane];
        iek = global(e.ierr + pix0)[(uint32_t)lane];
    }
    double rd = (double)r;

    // pass 1 of one visit: the term, and whether a lane is inside the cutoff
    auto term = [&](const HotGauss &H, const float2 &L, uint64_t &in_lanes) {
        float dx = x - H.xcen, dy = y - H.ycen, vx, vy;
        if (CENTRE) {   // the pixel offset from the FP64 centre
            dx -= L.x;
            dy -= L.y;
        }
        const float ea = exponent1(dx, dy, H.sfxx, H.sfyy, H.sfxy, vx, vy);
        const bool in = !(ea < kCutScaled);
        in_lanes = __builtin_amdgcn_ballot_w64(in);
        const float gp = cut_exp(in, ea);
        return H.ampA * gp * fmaf(vx, vx, fmaf(vy, vy, H.hcs));
    };
    auto subtract_bright = [&](float c, const HotGauss &H, float tb) {
        if (__builtin_amdgcn_ballot_w64(fabsf(c) > tb) == 0) {
            rd -= (double)c;
            return;
        }
        // FP64 copies of the coordinates made here: kept across the loop they
        // would hold 4 more registers
        float xb = x, yb = y;
        asm volatile("" : "+v"(xb), "+v"(yb));
        const double b = minus_value64(
            rd, g64[__builtin_amdgcn_readfirstlane(H.tag)], xb, yb);
        rd = fabsf(c) > tb ? b : rd - (double)c;
    };

    __shared__ HotGauss rec[kWave];
    __shared__ float2 rec_lo[CENTRE ? kWave : 1];
    HotGauss h;   // lane j: Gaussian base + j
    float2 h_lo = {0.0f, 0.0f};
    auto fetch = [&](int j) {
        const uint32_t i = min(j, ng - 1);
        h = load_hot(hot + e.gauss_off, i);
        if (CENTRE) h_lo = {g[i].xcen_lo, g[i].ycen_lo};
    };
    fetch(lane);
    uint64_t *__restrict__ fl = flags + t.flag + k;
    for (int base = 0; base < ng; base += kWave, fl += K) {
        const int j = base + lane;
        bool hit =
            j < ng && (cull == 0 || meets(xlo - h.xcen, xhi - h.xcen, ylo - h.ycen,
                                          yhi - h.ycen, h.sfxx, h.sfyy, h.sfxy));
        const bool one_by_one = (far | __builtin_amdgcn_ballot_w64(h.tag != 0)) != 0;
        if (one_by_one) {
            if (cull != 0 && j < ng && (far != 0 || h.tag != 0))
                hit = !boxed_out(1, gboxes[e.gauss_off + j], box);
        }
        const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
        const int cnt = __builtin_popcountll(m);
        const int rank = rank_in(m);
        if (hit) {
            h.tag = j;
            rec[rank] = h;
            if (CENTRE) rec_lo[rank] = h_lo;
        }
        wave_lds_sync();
        fetch(j + kWave);   // the next block's, under this block's visits
        // bit cnt - 1 - n of act: the n-th visit had a lane inside the cutoff
        // (shifted in through the scalar carry: two additions of act to itself)
        uint32_t act_lo = 0, act_hi = 0;
        auto note = [&](uint64_t in_lanes) {
            asm("s_cmp_lg_u64 %2, 0\n\ts_addc_u32 %0, %0, %0\n\ts_addc_u32 %1, %1, %1"
                : "+s"(act_lo), "+s"(act_hi)
                : "s"(in_lanes)
                : "scc");
        };
        const int together = one_by_one ? 0 : cnt - cnt % kVisits;
        int n = 0;
        for (; n < together; n += kVisits) {
            HotGauss H[kVisits];
            float2 L[kVisits];
            float c[kVisits], top = 0.0f;
#pragma unroll
            for (int u = 0; u < kVisits; ++u) {
                H[u] = rec[n + u];
                if (CENTRE) L[u] = rec_lo[n + u];
            }
            __builtin_amdgcn_sched_barrier(0);   // all loads before the first wait
#pragma unroll
            for (int u = 0; u < kVisits; ++u) {
                uint64_t in_lanes;
                c[u] = term(H[u], L[u], in_lanes);
                note(in_lanes);
                if (MIXED) top = fmaxf(top, fabsf(c[u]));
            }
            if (!MIXED) {
#pragma unroll
                for (int u = 0; u < kVisits; ++u) r -= c[u];
            } else if (__builtin_amdgcn_ballot_w64(top > t.tmin) == 0) {
#pragma unroll
                for (int u = 0; u < kVisits; ++u) rd -= (double)c[u];
            } else {
#pragma unroll
                for (int u = 0; u < kVisits; ++u) subtract_bright(c[u], H[u], t.tmin);
            }
        }
        for (; n < cnt; ++n) {
            const HotGauss H = rec[n];
            uint64_t in_lanes;
            const float c = term(H, CENTRE ? rec_lo[n] : float2{0.0f, 0.0f}, in_lanes);
            note(in_lanes);
            float tb = t.tmin;
            if (one_by_one) {
                if (in_lanes == 0) continue;
                if (MIXED && !(g[__builtin_amdgcn_readfirstlane(H.tag)].peak > t.tmin))
                    tb = __builtin_huge_valf();
            }
            if (MIXED)
                subtract_bright(c, H, tb);
            else
                r -= c;
        }
        wave_lds_sync();   // before the next block's records
        const uint64_t act = (uint64_t)act_hi << 32 | act_lo;
        const uint64_t word = __builtin_amdgcn_ballot_w64(
            hit && ((act >> ((cnt - 1 - rank) & 63)) & 1));
        if (lane == 0) *fl = word;
    }
    if (!MIXED) rd = (double)r;
    r = (float)rd;
    const uint32_t o = (uint32_t)(t.chunk0 + k) * kWave + lane;
    resid[o] = rd;
    weight[o] = -2.0f * ((r * iek) * iek);   // -2 r ierr^2
    if (e.residual != nullptr && lane < npix) e.residual[pix0 + lane] = r;
}

// Pass 2 of one source of one tile, or (source n_src) the tile's chi2.
template <int K, bool MIXED, bool CENTRE>
__global__ __launch_bounds__(kWave) FPHO_EVAL_OCCUPANCY void gradient_kernel(
    const TileDesc *__restrict__ tiles, const int2 *__restrict__ items,
    const ExpDesc *__restrict__ exps, const ImgGauss *__restrict__ gauss,
    const uint64_t *__restrict__ flags, const double *__restrict__ resid,
    const float *__restrict__ weight, float *__restrict__ gpart, double *__restrict__ cpart) {
    const int lane = threadIdx.x;
    const int2 item = items[xcd_rotate((int)blockIdx.x, (int)gridDim.x, 0)];
    const int tile = item.x, s = item.y;
    const TileDesc t = tiles[tile];
    const ExpDesc &e = exps[t.exp];
    const uint32_t slot = (uint32_t)t.chunk0 * kWave;
    if (s == e.n_src) {
        // sum (r^2 - d^2) ierr^2 (compute_gaussians_kernel.cu:276-287)
        double c2 = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t p = k * kWave + lane;
            float dk = 0.0f, iek = 0.0f;
            double rd = 0.0;
            if ((int)p < t.npix) {
                dk = global(e.data + t.pix0)[p];
                iek = global(e.ierr + t.pix0)[p];
                rd = resid[slot + p];
            }
            c2 = add_chi2<MIXED>(c2, rd, dk, iek);
        }
        c2 = wave_sum(c2);
        if (lane == 0) cpart[tile] = c2;
        return;
    }
    float x[K], y[K], rr[K];
    if (t.npix == K * kWave) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t p = k * kWave + lane;
            x[k] = global(e.xpix + t.pix0)[p] - e.x0;
            y[k] = global(e.ypix + t.pix0)[p] - e.y0;
            rr[k] = (weight + slot)[p];
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t p = k * kWave + lane;
            x[k] = y[k] = kMaskedCoord;
            rr[k] = 0.0f;
            if ((int)p < t.npix) {
                x[k] = global(e.xpix + t.pix0)[p] - e.x0;
                y[k] = global(e.ypix + t.pix0)[p] - e.y0;
                rr[k] = (weight + slot)[p];
            }
        }
    }
    const ImgGauss *__restrict__ g = gauss + e.gauss_off;
    const uint32_t *__restrict__ fl = reinterpret_cast<const uint32_t *>(flags + t.flag);
    const int n_psf = e.n_psf;
    __shared__ HotGauss rec[kWave];
    SourcePartials src;
    bool touched = false;
    for (int cb = 0; cb < n_psf; cb += kWave) {
        // lane l: the slots in which Gaussian i is active
        const bool valid = cb + lane < n_psf;
        const uint32_t i = s * n_psf + (valid ? cb + lane : 0);
        uint32_t mask = 0;
        if (valid) {
            const uint32_t f = (i >> 6) * (2 * K) + ((i >> 5) & 1);
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (k * kWave < t.npix) mask |= ((fl[f + 2 * k] >> (i & 31)) & 1) << k;
        }
        const uint64_t m = __builtin_amdgcn_ballot_w64(mask != 0);
        const int cnt = __builtin_popcountll(m);
        if (cnt == 0) continue;
        touched = true;
        if (mask != 0) {
            // from the full record, so that its line is in the L2 when the
            // epilogue's scalar loads come (against the short records: 16 tiles
            // of 54 Gaussians 53.7 -> 52.2 us a pass)
            HotGauss h = load_record(g, i);
            h.tag = i << 8 | mask;
            rec[rank_in(m)] = h;
        }
        wave_lds_sync();
        for (int n = 0; n < cnt; ++n) {
            const HotGauss H = rec[n];
            const uint32_t v = __builtin_amdgcn_readfirstlane(H.tag);
            const ImgGauss &G = g[v >> 8];
            const float xcl = CENTRE ? G.xcen_lo : 0.0f, ycl = CENTRE ? G.ycen_lo : 0.0f;
            GradSums q;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (!(v & (1u << k))) continue;
                float dx = x[k] - H.xcen, dy = y[k] - H.ycen;
                if (CENTRE) {
                    dx -= xcl;
                    dy -= ycl;
                }
                q.add(dx, dy, rr[k], H.sfxx, H.sfyy, H.sfxy, H.hcs);
            }
            src.add(G, H.sfxx, H.sfyy, H.sfxy, q);
        }
        wave_lds_sync();   // before the next 64 Gaussians' records
    }
    float *o = gpart + t.part_off + kNParams * s;
    if (touched)
        src.write(o, e.CW + 4 * s, lane);
    else if (lane < kNParams)
        o[lane] = 0.0f;
}

// The gradient launch's waves.  A run is the tiles of one exposure that stand
// together in the queue; its items go source by source, tile by
// tile, so waves that run together read the same records from the scalar
// caches (10 bands x 9 exposures, 13 sources: 1071 -> 1023 us a pass against
// tile by tile).  The short chi2 waves go behind all others: at the end of their
// run they met the same CUs in every run of a plan with few sources (256
// exposures of 64^2, one source, K = 4: 95 us a pass, 79 with one wave per tile).
// runs[q]: first item, place in the run and its length.
__global__ __launch_bounds__(256) void list_items_kernel(
    const TileDesc *__restrict__ tiles, const int32_t *__restrict__ queue,
    const ExpDesc *__restrict__ exps, const int4 *__restrict__ runs, int32_t n_tiles,
    int32_t n_items, int2 *__restrict__ items) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n_tiles) return;
    const int tile = queue[q], n_src = exps[tiles[tile].exp].n_src;
    const int4 r = runs[q];
    for (int s = 0; s < n_src; ++s) items[r.x + s * r.z + r.y] = make_int2(tile, s);
    items[n_items - n_tiles + q] = make_int2(tile, n_src);
}

__global__ void zero_counter_kernel(int32_t *counter) {
    if (threadIdx.x == 0 && blockIdx.x == 0) counter[0] = 0;
}

// ------------------------------------------------------------------ reduce

// Workgroups (patch-band, 64 columns).  Column j of the band's [ntiles][n_src*7]
// partial block is cut into S segments of consecutive tiles, S a function of
// the column count only (S * ncol <= kReduceSlots); each segment is summed in
// tile order by one lane, then each column's S segment sums in segment
// order.  chi2 partials go through a fixed-shape tree (first column group).
// The result depends only on (ntiles, ncol), not on tile execution order or
// the launch.  Bound by load latency: a single patch has few (patch, band)
// groups, so the columns are spread over workgroups and a lane keeps 16 loads
// in flight (us, one workgroup and 4 loads -> these: 12 bands x 512 tiles x
// 420 columns 24.0 -> 6.2; 10 x 2304 x 91 28.6 -> 12.7; 96 patches 41 -> 26).
constexpr int kReduceSlots = 4096;
constexpr int kReduceCols = 64;        // columns per workgroup
constexpr int kReduceSegs = 16;        // S at most
constexpr int kReduceThreads = kReduceCols * kReduceSegs;

template <typename Acc>
__global__ __launch_bounds__(kReduceThreads) void reduce_kernel(
    const OutDesc *__restrict__ outs, const float *__restrict__ gpart,
    const double *__restrict__ cpart, double *__restrict__ chi2,
    double *__restrict__ dchi2) {
    __shared__ Acc seg[kReduceThreads];
    __shared__ Acc sh[kReduceThreads];
    const OutDesc o = outs[blockIdx.x];
    const int ncol = o.n_src * kNParams;
    const int j0 = blockIdx.y * kReduceCols;
    if (j0 >= ncol) return;
    const int S = max(1, min(kReduceSegs, kReduceSlots / ncol));
    const int len = (o.ntiles + S - 1) / S;   // tiles per segment
    const int j = j0 + threadIdx.x % kReduceCols, r = threadIdx.x / kReduceCols;
    if (j < ncol && r < S) {
        const int t0 = r * len, t1 = min(o.ntiles, t0 + len);
        const float *col = gpart + o.part0 + j;
        Acc acc = 0;
        int t = t0;
        for (; t + 16 <= t1; t += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = col[(int64_t)(t + u) * ncol];
#pragma unroll
            for (int u = 0; u < 16; ++u) acc += (Acc)v[u];
        }
#pragma unroll 4
        for (; t < t1; ++t) acc += (Acc)col[(int64_t)t * ncol];
        seg[threadIdx.x] = acc;
    }
    Acc c = 0;
    if (j0 == 0)
        for (int t = threadIdx.x; t < o.ntiles; t += kReduceThreads) c += (Acc)cpart[o.tile0 + t];
    sh[threadIdx.x] = c;
    __syncthreads();
    if (r == 0 && j < ncol) {
        Acc acc = 0;
        for (int q = 0; q < S; ++q) acc += seg[q * kReduceCols + threadIdx.x];
        dchi2[o.dchi2_out + j] = (double)acc;
    }
    if (j0 > 0) return;
    for (int w = kReduceThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) chi2[o.chi2_out] = (double)sh[0];
}

// ------------------------------------------------- proposals from parameters

// Cubic B-spline basis on knot span l (t[l] <= x < t[l+1]): N[0..3] are the
// values of N_{l-3..l,3}(x), dN their derivatives (Cox-de Boor recursion).
__device__ inline void bspline3(const double *t, int l, double x, double N[4],
                                double dN[4]) {
    double left[4], right[4], N2[3];
    N[0] = 1.0;
    for (int j = 1; j <= 3; ++j) {
        left[j] = x - t[l + 1 - j];
        right[j] = t[l + j] - x;
        double saved = 0.0;
        for (int r = 0; r < j; ++r) {
            const double tmp = N[r] / (right[r + 1] + left[j - r]);
            N[r] = saved + right[r + 1] * tmp;
            saved = left[j - r] * tmp;
        }
        N[j] = saved;
        if (j == 2) {
            N2[0] = N[0];
            N2[1] = N[1];
            N2[2] = N[2];
        }
    }
    // d/dx N_{i,3} = 3 (N_{i,2}/(t[i+3]-t[i]) - N_{i+1,2}/(t[i+4]-t[i+1])),
    // N2[r] = N_{l-2+r,2}; N_{l-3,2} = N_{l+1,2} = 0 on this span.
    for (int r = 0; r < 4; ++r) {
        const int i = l - 3 + r;
        const double a = (r >= 1) ? N2[r - 1] / (t[i + 3] - t[i]) : 0.0;
        const double b = (r <= 2) ? N2[r] / (t[i + 4] - t[i + 1]) : 0.0;
        dN[r] = 3.0 * (a - b);
    }
}

__device__ inline int knot_span(const double *t, int n_t, double x) {
    // largest l in [3, n_t-5] with t[l] <= x  (x already clamped)
    int lo = 3, hi = n_t - 5;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (t[mid] <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// One wave per source: lane m evaluates mixture component m, and the wave
// writes the FP32 record to props and/or the FP64 record to props64 (either
// may be null).  Bound by the latency of the knot search and of a component's
// 16 coefficients; one lane per source ran the components one after another
// (us, before -> after: four patches 10.7 -> 4.7, 96 patches 21.5 -> 7.2).
__global__ __launch_bounds__(kWave) void theta_kernel(
    const SrcDesc *__restrict__ srcs, const double *__restrict__ theta, SplineView sp,
    fpho_source *__restrict__ props, Source64 *__restrict__ props64,
    uint32_t *__restrict__ status) {
    const int lane = threadIdx.x;
    const SrcDesc sd = srcs[blockIdx.x];
    const double *th = theta + sd.theta_off;
    const int nb = sd.n_bands;
    const double v = lane < nb + 6 ? th[lane] : 0.0;   // nb + 6 <= 36
    if (__builtin_amdgcn_ballot_w64(!isfinite(v)) != 0 && lane == 0)
        atomicOr(status, FPHO_STATUS_THETA_NONFINITE);
    const double n = th[nb + 4], rh = th[nb + 5];

    double amp = 0.0, amp_n = 0.0, amp_r = 0.0;   // component `lane`
    if (n < sp.nsersic_min) {
        // one-hot at the radius closest to rh (forcepho/sources.py:662-665)
        int best = 0;
        double bd = fabs(rh - sp.radii[0]);
        for (int m = 1; m < sp.n_amp; ++m) {
            const double dd = fabs(rh - sp.radii[m]);
            if (dd < bd) {
                bd = dd;
                best = m;
            }
        }
        amp = lane == best ? 1.0 : 0.0;
    } else if (rh < 0.0) {
        amp = lane == 0 ? 1.0 : 0.0;  // forcepho/sources.py:666-668
    } else {
        const double xn = fmin(fmax(n, sp.tx[3]), sp.tx[sp.n_tx - 4]);
        const double xr = fmin(fmax(rh, sp.ty[3]), sp.ty[sp.n_ty - 4]);
        const int lx = knot_span(sp.tx, sp.n_tx, xn);
        const int ly = knot_span(sp.ty, sp.n_ty, xr);
        double Nx[4], dNx[4], Ny[4], dNy[4];
        bspline3(sp.tx, lx, xn, Nx, dNx);
        bspline3(sp.ty, ly, xr, Ny, dNy);
        const int ny = sp.n_ty - 4;
        const int nx = sp.n_tx - 4;
        if (lane < sp.n_amp) {
            const double *c = sp.coeffs + (int64_t)lane * nx * ny;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const double *row = c + (int64_t)(lx - 3 + a) * ny + (ly - 3);
                double rv = 0.0, rd = 0.0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    rv += row[b] * Ny[b];
                    rd += row[b] * dNy[b];
                }
                amp += Nx[a] * rv;
                amp_n += dNx[a] * rv;
                amp_r += Nx[a] * rd;
            }
        }
    }
    // fields in record order: ra, dec, q, pa, nsersic, rh, then the arrays
    const double shape = lane < 6 ? th[nb + lane] : 0.0;
    const double flux = lane < nb ? v : 0.0;
    if (props64) {
        Source64 &o = props64[sd.proposal];
        if (lane < 6) (&o.ra)[lane] = shape;
        if (lane < FPHO_MAXBANDS) o.fluxes[lane] = flux;
        if (lane < FPHO_MAXRADII) {
            o.mixture_amplitudes[lane] = amp;
            o.damplitude_drh[lane] = amp_r;
            o.damplitude_dnsersic[lane] = amp_n;
        }
    }
    if (props) {
        fpho_source &f = props[sd.proposal];
        if (lane < 6) (&f.ra)[lane] = (float)shape;
        if (lane < FPHO_MAXBANDS) f.fluxes[lane] = (float)flux;
        if (lane < FPHO_MAXRADII) {
            f.mixture_amplitudes[lane] = (float)amp;
            f.damplitude_drh[lane] = (float)amp_r;
            f.damplitude_dnsersic[lane] = (float)amp_n;
        }
    }
}

// ------------------------------------------------------- gradient stacking

// One wave per source (lane: parameter of its block), then one lane per patch.
// Latency bound: a lane's loads over the bands are independent, the bands are
// added in order (us, one lane per source -> one wave: four patches 5.9 ->
// 4.6, 96 patches 12.6 -> 4.8).
__global__ __launch_bounds__(kWave) void stack_kernel(
    const SrcDesc *__restrict__ srcs, int32_t n_srcs, const PatchOut *__restrict__ pouts,
    int32_t n_patches, const double *__restrict__ chi2, const double *__restrict__ dchi2,
    double *__restrict__ lnlike, double *__restrict__ grad) {
    const int lane = threadIdx.x;
    if ((int)blockIdx.x < n_srcs) {
        const SrcDesc sd = srcs[blockIdx.x];
        const double *dv = dchi2 + sd.dchi2_base;
        const int nb = sd.n_bands;
        if (lane < nb) {
            grad[sd.theta_off + lane] = -0.5 * dv[(int64_t)lane * sd.src_stride];
        } else if (lane < nb + kNParams - 1) {
            const double *col = dv + lane - nb + 1;
            double acc = 0.0;
#pragma unroll 4
            for (int b = 0; b < nb; ++b) acc += col[(int64_t)b * sd.src_stride];
            grad[sd.theta_off + lane] = -0.5 * acc;
        }
        return;
    }
    const int i = ((int)blockIdx.x - n_srcs) * kWave + lane;
    if (i < n_patches) {
        const PatchOut po = pouts[i];
        double acc = 0.0;
#pragma unroll 4
        for (int b = 0; b < po.n_bands; ++b) acc += chi2[po.chi2_off + b];
        lnlike[i] = -0.5 * acc;
    }
}

// ------------------------------------------------- bounded transform, leapfrog

__device__ __forceinline__ double sigmoid(double z) { return 1.0 / (1.0 + exp(-z)); }

// One parameter a lane; see fpho_step.  Launch bound: it stands for the 22
// elementwise torch kernels of 4.6 us each that a leapfrog step took (8 patches
// of 32 sources, 10 steps: 4930 -> 4420 us a trajectory).  Every operation is
// rounded by itself and in their order, so no bit changes.
__global__ __launch_bounds__(kWave) void step_kernel(const fpho_step s) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * kWave + threadIdx.x;
    if (i >= s.n) return;
    double z = s.z[i];
    double y = sigmoid(z);
    const double range = s.range[i];
    double g = 0.0;
    if (s.grad_q) {
        const double jac = range * y * (1.0 - y);
        g = s.grad_q[i] * jac + (1.0 - 2.0 * y);
        if (s.grad) s.grad[i] = g;
    } else if (s.grad) {
        g = s.grad[i];
    }
    if (s.lnjac) {
        const double a = fabs(z);
        s.lnjac[i] = s.log_range[i] - a - 2.0 * log1p(exp(-a));
    }
    if (s.p) {
        const double eps = s.eps[i];
        const double p = s.p[i] + s.kick * eps * g;
        s.p_out[i] = p;
        if (s.z_out) {
            z = z + eps * (s.inv_mass[i] * p);
            s.z_out[i] = z;
            y = sigmoid(z);
        }
    }
    if (s.q_out) s.q_out[i] = s.lower[i] + y * range;
}

// ------------------------------------------------------ compat Response out

// dchi2 [n_bands][n_src][7] (double) -> Response[n_bands] (float, stride
// MAXSOURCES * 7, compute_gaussians_kernel.cu:304-310), tail zeroed.
__global__ __launch_bounds__(256) void response_kernel(const double *__restrict__ dchi2,
                                                       int32_t n_src,
                                                       fpho_response *__restrict__ out) {
    const int b = blockIdx.x;
    constexpr int kStride = FPHO_MAXSOURCES * kNParams;
    for (int j = threadIdx.x; j < kStride; j += blockDim.x)
        out[b].dchi2_dparam[j] =
            j < n_src * kNParams ? (float)dchi2[(int64_t)b * n_src * kNParams + j] : 0.0f;
}

// ---------------------------------------------------------------- launchers

template <typename Src>
static hipError_t launch_convert_t(const ExpDesc *exps, int64_t n_exp, int32_t max_ng, const Src *props,
                                   ImgGauss *out, ImgGauss64 *out64, int4 *boxes, HotGauss *hot,
                                   uint32_t *status, hipStream_t stream) {
    if (n_exp <= 0) return hipSuccess;
    // a wave per 64 Gaussians until there are 16384 waves (64 per CU)
    const int64_t blocks = std::max(1, (max_ng + kWave - 1) / kWave);
    const int64_t parts = std::min(blocks, std::max<int64_t>(1, 16384 / n_exp));
    hipLaunchKernelGGL(convert_kernel<Src>, dim3((unsigned)n_exp, (unsigned)parts), dim3(kWave),
                       0, stream, exps, props, out, out64, boxes, hot, status);
    return hipGetLastError();
}

hipError_t launch_convert(const ExpDesc *exps, int64_t n_exp, int32_t max_ng,
                          const fpho_source *props,
                          ImgGauss *out, ImgGauss64 *out64, int4 *boxes, HotGauss *hot,
                          uint32_t *status, hipStream_t stream) {
    return launch_convert_t(exps, n_exp, max_ng, props, out, out64, boxes, hot, status, stream);
}

hipError_t launch_convert(const ExpDesc *exps, int64_t n_exp, int32_t max_ng,
                          const Source64 *props,
                          ImgGauss *out, ImgGauss64 *out64, int4 *boxes, HotGauss *hot,
                          uint32_t *status, hipStream_t stream) {
    return launch_convert_t(exps, n_exp, max_ng, props, out, out64, boxes, hot, status, stream);
}

hipError_t launch_response(const double *dchi2, int32_t n_bands, int32_t n_src,
                           fpho_response *out, hipStream_t stream) {
    if (n_bands <= 0) return hipSuccess;
    hipLaunchKernelGGL(response_kernel, dim3((unsigned)n_bands), dim3(256), 0, stream, dchi2,
                       n_src, out);
    return hipGetLastError();
}

template <int K, bool MIXED, bool CENTRE>
static hipError_t launch_eval_k(const EvalArgs &a, hipStream_t stream) {
    if (a.n_items > 0) {
        hipLaunchKernelGGL((residual_kernel<K, MIXED, CENTRE>), dim3((unsigned)(K * a.n_tiles)),
                           dim3(kWave), 0, stream, a.tiles, a.queue, a.exps, a.gauss, a.gauss64,
                           a.hot, a.gboxes, a.slot_boxes, a.flags, a.resid, a.weight,
                           (int32_t)a.cull);
        hipLaunchKernelGGL((gradient_kernel<K, MIXED, CENTRE>), dim3((unsigned)a.n_items),
                           dim3(kWave), 0, stream, a.tiles, a.items, a.exps, a.gauss, a.flags,
                           a.resid, a.weight, a.gpart, a.cpart);
        return hipGetLastError();
    }
    const int W = a.waves_per_group;
    // per wave: 64 records, the slot mask bytes, then the activity words
    const size_t lds = (size_t)W * (kWave * sizeof(HotGauss) + (size_t)a.mask_cap +
                                    8 * (size_t)a.act_words);
    if (a.persistent) {
        hipLaunchKernelGGL(zero_counter_kernel, dim3(1), dim3(64), 0, stream, a.counter);
        hipLaunchKernelGGL((eval_persistent_kernel<K, MIXED, CENTRE>), dim3((unsigned)a.grid),
                           dim3(64 * W), lds, stream, a.tiles, a.queue, (int32_t)a.n_tiles,
                           a.counter, a.exps, a.gauss, a.gauss64, a.gboxes, a.slot_boxes, a.gpart, a.cpart,
                           (int32_t)a.cull, (int32_t)a.mask_cap, (int32_t)a.act_words);
    } else {
        const int64_t groups = (a.n_tiles + W - 1) / W;
        hipLaunchKernelGGL((eval_kernel<K, MIXED, CENTRE>), dim3((unsigned)groups), dim3(64 * W), lds,
                           stream, a.tiles, a.queue, (int32_t)a.n_tiles, (int32_t)W, a.exps,
                           a.gauss, a.gauss64, a.gboxes, a.slot_boxes, a.gpart, a.cpart, (int32_t)a.cull,
                           (int32_t)a.mask_cap, (int32_t)a.act_words);
    }
    return hipGetLastError();
}

template <bool MIXED, bool CENTRE>
static hipError_t launch_eval_p(const EvalArgs &a, hipStream_t stream) {
    switch (a.pix_per_lane) {
        case 1: return launch_eval_k<1, MIXED, CENTRE>(a, stream);
        case 2: return launch_eval_k<2, MIXED, CENTRE>(a, stream);
        case 4: return launch_eval_k<4, MIXED, CENTRE>(a, stream);
        case 8: return launch_eval_k<8, MIXED, CENTRE>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_eval(const EvalArgs &a, hipStream_t stream) {
    if (a.n_tiles <= 0) return hipSuccess;
    switch (a.precision) {
        case kPrecMixed: return launch_eval_p<true, false>(a, stream);
        case kPrecMixedCentre: return launch_eval_p<true, true>(a, stream);
        default: return launch_eval_p<false, false>(a, stream);
    }
}

hipError_t launch_list_items(const TileDesc *tiles, const int32_t *queue, const ExpDesc *exps,
                             const int4 *runs, int64_t n_tiles, int64_t n_items, int2 *items,
                             hipStream_t stream) {
    if (n_tiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(list_items_kernel, dim3((unsigned)((n_tiles + 255) / 256)), dim3(256), 0,
                       stream, tiles, queue, exps, runs, (int32_t)n_tiles, (int32_t)n_items, items);
    return hipGetLastError();
}

hipError_t launch_reduce(const OutDesc *outs, int64_t n_outs, int32_t max_src, const float *gpart,
                         const double *cpart, double *chi2, double *dchi2, int fp64,
                         hipStream_t stream) {
    if (n_outs <= 0) return hipSuccess;
    const dim3 grid((unsigned)n_outs,
                    (unsigned)((max_src * kNParams + kReduceCols - 1) / kReduceCols));
    if (fp64)
        hipLaunchKernelGGL(reduce_kernel<double>, grid, dim3(kReduceThreads), 0, stream, outs,
                           gpart, cpart, chi2, dchi2);
    else
        hipLaunchKernelGGL(reduce_kernel<float>, grid, dim3(kReduceThreads), 0, stream, outs,
                           gpart, cpart, chi2, dchi2);
    return hipGetLastError();
}

hipError_t launch_theta(const SrcDesc *srcs, int64_t n_srcs, const double *theta,
                        const SplineView &sp, fpho_source *props, Source64 *props64,
                        uint32_t *status, hipStream_t stream) {
    if (n_srcs <= 0) return hipSuccess;
    hipLaunchKernelGGL(theta_kernel, dim3((unsigned)n_srcs), dim3(kWave), 0, stream, srcs, theta,
                       sp, props, props64, status);
    return hipGetLastError();
}

hipError_t launch_stack(const SrcDesc *srcs, int64_t n_srcs, const PatchOut *pouts,
                        int64_t n_patches, const double *chi2, const double *dchi2,
                        double *lnlike, double *grad, hipStream_t stream) {
    const int64_t n = n_srcs + (n_patches + kWave - 1) / kWave;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(stack_kernel, dim3((unsigned)n), dim3(kWave), 0, stream, srcs, (int32_t)n_srcs,
                       pouts, (int32_t)n_patches, chi2, dchi2, lnlike, grad);
    return hipGetLastError();
}

hipError_t launch_step(const fpho_step &s, hipStream_t stream) {
    if (s.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(step_kernel, dim3((unsigned)((s.n + kWave - 1) / kWave)), dim3(kWave), 0,
                       stream, s);
    return hipGetLastError();
}

}  // namespace fpho
