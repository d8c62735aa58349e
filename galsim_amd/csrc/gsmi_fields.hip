// Parameter maps of the differentiable Exponential (x) Moffat model, fused into one kernel each
// way: parameter rows -> the lowered records' fields (written straight into the device records),
// and field gradients -> parameter gradients (the chain rule).  They restate on the device what
// the host lowering does with galsim/exponential.py (r0 = hlr / 1.6783469900166605),
// galsim/shear.py:365-386 (the shear matrix), galsim/moffat.py (rD from fwhm and beta) and the
// Moffat normalisation of src/SBMoffat.cpp:226-243; nothing here replaces a reference entry
// point.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "../../include/gsmi.h"
#include "launch.h"

namespace gsmi {
namespace {

constexpr int kF = GSMI_GRAD_FIELDS;
constexpr int kP = GSMI_GRAD_PER_LEAF;
constexpr int kUX = kP * GSMI_GRAD_MAXLEAF;
constexpr double kHlrToR0 = 1.6783469900166605;   // Exponential hlr / r0

// psi(x), x > 0: the recurrence psi(x) = psi(x + 1) - 1/x up to x >= 10, then the asymptotic
// series of Abramowitz & Stegun 6.3.18 (terms to x^-12; truncation < 1e-16 at x = 10).
__device__ double digamma(double x)
{
    double r = 0.;
    while (x < 10.) {
        r -= 1. / x;
        x += 1.;
    }
    const double i2 = 1. / (x * x);
    const double s = i2 * (1. / 12. - i2 * (1. / 120. - i2 * (1. / 252. - i2 * (1. / 240. -
                     i2 * (1. / 132. - i2 * (691. / 32760.))))));
    return r + log(x) - 0.5 / x - s;
}

// Field k of theta row (flux, hlr, g1, g2, dx, dy, psf_fwhm [, beta]); base where no parameter
// reaches.
__device__ double field_of(const double* th, int k, bool fit_beta, double base, double cx,
                           double cy, double inv_scale, double fwhm_to_rd)
{
    if (k >= 2 && k <= 5) {
        const double g1 = th[2], g2 = th[3];
        const double a = inv_scale / sqrt(1. - (g1 * g1 + g2 * g2));
        return a * (k == 2 ? 1. + g1 : k == 5 ? 1. - g1 : g2);
    }
    switch (k) {
      case 0: return th[0];
      case 1: return th[1] / kHlrToR0;
      case kP + 1:
        return fit_beta ? th[6] / (2. * sqrt(pow(2., 1. / th[7]) - 1.)) : th[6] * fwhm_to_rd;
      case kP + 6: return fit_beta ? th[7] : base;   // (kP with beta free: the caller's)
      case kUX: return th[4] + cx;
      case kUX + 1: return th[5] + cy;
    }
    return base;
}

// 32 lanes per stamp, one per field: its table of 31 destinations and base values is read and the
// record written in whole lines, and the elementary functions run side by side.  A thread per
// stamp spent 14 us (23 us with beta free) on 1024 stamps in that chain.
//
// With beta free (nu = beta - 1) the record also holds, on the k^nu K_nu form, the flux
// 4 / (Gamma(nu) 2^beta) and the five values that follow beta: the k = 0 value 2^(nu-1) Gamma(nu)
// and the order-only constants of Temme's series for mu = nu - round(nu) (fact gam1, fact gam2,
// 1 / (2 Gamma(1+mu)), 1 / (2 Gamma(1-mu))), as moffat.temme_constants.  Lanes 0 to 2 take the
// three log-Gammas in one call, 0 to 3 the exponentials in one, and shuffles share them.
static_assert(kF <= 32, "a lane per field");
__global__ void __launch_bounds__(256)
exp_moffat_fields_kernel(const double* __restrict__ theta, int n, int fit_beta,
                         const double* __restrict__ base, const double* __restrict__ cxcy,
                         double inv_scale, const double* __restrict__ fwhm_to_rd,
                         const int64_t* __restrict__ dst, const int64_t* __restrict__ aux_dst,
                         double* __restrict__ records)
{
    const int i = blockIdx.x * (blockDim.x / 32) + threadIdx.x / 32;
    const int k = threadIdx.x % 32;
    if (i >= n) return;
    const double* th = theta + size_t(i) * (fit_beta ? 8 : 7);
    double mflux = 0.;
    if (fit_beta) {
        const double nu = th[7] - 1.;
        const double mu = nu - floor(nu + 0.5);
        const double lg = lgamma(k == 1 ? 1. + mu : k == 2 ? 1. - mu : nu);
        const double ex = exp(k == 0 ? (nu - 1.) * M_LN2 + lg :
                              k == 3 ? -lg - th[7] * M_LN2 : -lg);
        const double at0 = __shfl(ex, 0, 32), gampl = __shfl(ex, 1, 32),
                     gammi = __shfl(ex, 2, 32);
        mflux = 4. * __shfl(ex, 3, 32);
        if (aux_dst && k < 5) {
            const bool small = fabs(mu) < 1e-4;
            const double m2 = mu * mu;
            const double gam1 = small ? -(0.5772156649015329 - 0.0420026350340952 * m2)
                                      : (gammi - gampl) / (2. * mu);
            const double gam2 = small ? 1. - 0.6558780715202538 * m2 + 0.1665386113822915 * m2 * m2
                                      : (gammi + gampl) / 2.;
            const double fact = small ? 1. + (M_PI * mu) * (M_PI * mu) / 6.
                                      : M_PI * mu / sin(M_PI * mu);
            const double v = k == 0 ? at0 : k == 1 ? fact * gam1 : k == 2 ? fact * gam2 :
                             k == 3 ? 0.5 / gampl : 0.5 / gammi;
            records[aux_dst[size_t(i) * 5 + k]] = v;
        }
    }
    if (k < kF) {
        const int64_t d = dst[size_t(i) * kF + k];
        if (d >= 0)
            records[d] = fit_beta && k == kP
                             ? mflux
                             : field_of(th, k, fit_beta != 0, base[size_t(i) * kF + k],
                                        cxcy[2 * i], cxcy[2 * i + 1], inv_scale,
                                        fit_beta ? 0. : fwhm_to_rd[i]);
    }
}

// dL/dtheta from dL/dfields (rows in the plan's sorted order, inv[i] = row of stamp i).
__global__ void __launch_bounds__(256)
exp_moffat_grad_kernel(const double* __restrict__ theta, int n, int fit_beta,
                       const double* __restrict__ fwhm_to_rd, const double* __restrict__ gfields,
                       const int64_t* __restrict__ inv, double inv_scale,
                       double* __restrict__ dtheta)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int ncol = fit_beta ? 8 : 7;
    const double* th = theta + size_t(i) * ncol;
    const double* G = gfields + size_t(inv[i]) * kF;
    double* out = dtheta + size_t(i) * ncol;
    const double g1 = th[2], g2 = th[3];
    const double den2 = 1. - (g1 * g1 + g2 * g2);
    const double a = inv_scale / sqrt(den2);          // d a / d g = a g / den2
    const double b = a / den2;
    out[0] = G[0];
    out[1] = G[1] / kHlrToR0;
    // f2 = a (1 + g1), f3 = f4 = a g2, f5 = a (1 - g1)
    out[2] = G[2] * (a + b * (1. + g1) * g1) + (G[3] + G[4]) * (b * g2 * g1) +
             G[5] * (-a + b * (1. - g1) * g1);
    out[3] = G[2] * (b * (1. + g1) * g2) + (G[3] + G[4]) * (a + b * g2 * g2) +
             G[5] * (b * (1. - g1) * g2);
    out[4] = G[kUX];
    out[5] = G[kUX + 1];
    if (fit_beta) {
        const double beta = th[7];
        const double p = pow(2., 1. / beta);
        const double s = sqrt(p - 1.);
        out[6] = G[kP + 1] / (2. * s);
        const double mflux = 4. * exp(-lgamma(beta - 1.) - beta * M_LN2);
        // d mflux / d beta = -mflux (psi(beta - 1) + ln 2); d rD / d beta = fw p ln2 / (4 s^3 b^2)
        out[7] = G[kP] * (-mflux * (digamma(beta - 1.) + M_LN2)) +
                 G[kP + 1] * (th[6] * p * M_LN2 / (4. * s * s * s * beta * beta)) + G[kP + 6];
    } else {
        out[6] = G[kP + 1] * fwhm_to_rd[i];
    }
}

}  // namespace
}  // namespace gsmi

using namespace gsmi;

extern "C" {

int gsmi_exp_moffat_fields(const double* theta, int n, int fit_beta, const double* base,
                           const double* cxcy, double inv_scale, const double* fwhm_to_rd,
                           const int64_t* dst, const int64_t* aux_dst, double* records,
                           void* stream)
{
    if (n < 0 || !theta || !base || !cxcy || !dst || !records || (!fit_beta && !fwhm_to_rd)) {
        set_error("gsmi_exp_moffat_fields: bad arguments");
        return GSMI_E_ARG;
    }
    if (n == 0) return GSMI_OK;
    hipLaunchKernelGGL(exp_moffat_fields_kernel, dim3((n + 7) / 8), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), theta, n, fit_beta, base, cxcy,
                       inv_scale, fwhm_to_rd, dst, aux_dst, records);
    return hip_check(hipGetLastError(), "exp_moffat_fields launch");
}

int gsmi_exp_moffat_grad(const double* theta, int n, int fit_beta, const double* fwhm_to_rd,
                         const double* gfields, const int64_t* inv, double inv_scale,
                         double* dtheta, void* stream)
{
    if (n < 0 || !theta || !gfields || !inv || !dtheta || (!fit_beta && !fwhm_to_rd)) {
        set_error("gsmi_exp_moffat_grad: bad arguments");
        return GSMI_E_ARG;
    }
    if (n == 0) return GSMI_OK;
    hipLaunchKernelGGL(exp_moffat_grad_kernel, dim3((n + 255) / 256), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), theta, n, fit_beta, fwhm_to_rd,
                       gfields, inv, inv_scale, dtheta);
    return hip_check(hipGetLastError(), "exp_moffat_grad launch");
}

}  // extern "C"
