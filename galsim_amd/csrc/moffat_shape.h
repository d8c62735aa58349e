// The order derivative of the Moffat transform, for the gradient in beta.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "device_math.h"

namespace gsmi {

// d/dnu [k^nu K_nu(k)] (nu = beta - 1 >= 0.1) in FP64: k^nu (ln k K_nu + dK_nu/dnu), the order
// derivative by a central difference with step 1e-4 (truncation ~1e-9 relative, rounding
// ~1e-12); at k = 0 the limit 2^(nu-1) Gamma(nu) (ln 2 + psi(nu)), psi by the difference of
// lgamma.
__device__ __noinline__ double moffat_dg_dnu(double nu, double k)
{
    const double h = 1e-4;
    if (k == 0.) {
        const double g0 = exp((nu - 1.) * M_LN2 + lgamma(nu));
        const double psi = (lgamma(nu + h) - lgamma(nu - h)) / (2. * h);
        return g0 * (M_LN2 + psi);
    }
    const double lk = log(k);
    const double kp = bessel_k(nu + h, k);
    const double km = bessel_k(nu - h, k);
    const double kn = bessel_k(nu, k);
    return exp(nu * lk) * (lk * kn + (kp - km) / (2. * h));
}

// The same derivative in FP32 from the integral K_nu(k) = int_0^inf exp(-k cosh t) cosh(nu t) dt
// (Abramowitz & Stegun 9.6.24), whose nu-derivative is int_0^inf t sinh(nu t) exp(-k cosh t) dt.
// With L = ln k both become sums over nodes t_m of e+ = exp(nu (t_m + L) - k cosh t_m) and
// e- = exp(nu (L - t_m) - k cosh t_m):  k^nu K_nu = sum w_m (e+ + e-) / 2 and
// d/dnu [k^nu K_nu] = sum w_m ((t_m + L) e+ + (L - t_m) e-) / 2, the trapezoid rule with step
// h = 11/32.  The integrands are analytic in |Im t| < pi/2 and decay double-exponentially, so
// the rule converges like exp(-pi^2 / h); measured against FP64 Bessel functions its error is
// below 1.2e-6 of the k = 0 value for nu <= 5.5 (3e-6 at nu = 8), over k in [1e-4, 60].  The sum
// stops once e+ is past its peak and below 1e-9 of the running sum (e- <= e+ throughout); at
// most 48 nodes (t <= 16.2, enough for k >= 1e-5).  L is split as e ln2_hi + (ln m + e ln2_lo)
// (k = m 2^e, m in [1/sqrt2, sqrt2)), so t_m + e ln2_hi is exact and L carries no rounding of
// its large part into the exponents.  k = 0 takes the FP64 limit.
__device__ inline float moffat_dg_dnu_f32(float nu, float k)
{
    if (k == 0.f) return float(moffat_dg_dnu(double(nu), 0.));
    constexpr float kCosh[48] = {
        1.000000000e+00f, 1.059666109e+00f, 1.245784524e+00f, 1.580565168e+00f, 2.103958159e+00f,
        2.878421143e+00f, 3.996372503e+00f, 5.591219856e+00f, 7.853279873e+00f, 1.105248919e+01f,
        1.557061655e+01f, 2.194682011e+01f, 3.094198637e+01f, 4.362952848e+01f, 6.152347897e+01f,
        8.675916262e+01f, 1.223480095e+02f, 1.725369157e+02f, 2.433150346e+02f, 3.431284761e+02f,
        4.838881994e+02f, 6.823913746e+02f, 9.623258256e+02f, 1.357096751e+03f, 1.913813041e+03f,
        2.698908885e+03f, 3.806071511e+03f, 5.367421090e+03f, 7.569276928e+03f, 1.067439137e+04f,
        1.505330460e+04f, 2.122856204e+04f, 2.993707087e+04f, 4.221803674e+04f, 5.953697455e+04f,
        8.396059155e+04f, 1.184034121e+05f, 1.669755744e+05f, 2.354733022e+05f, 3.320705813e+05f,
        4.682945791e+05f, 6.604012075e+05f, 9.313149763e+05f, 1.313364626e+06f, 1.852140989e+06f,
        2.611937444e+06f, 3.683422184e+06f, 5.194457862e+06f,
    };
    constexpr float h = 0.34375f;
    constexpr float kLog2e = 1.44269504088896341f;
    int ex;
    float mant = frexpf(k, &ex);
    if (mant < 0.70710678f) {
        mant *= 2.f;
        --ex;
    }
    const float eh = float(ex) * 0.693145751953125f;       // 12-bit constant: exact
    const float el = __logf(mant) + float(ex) * 1.428606765330187e-6f;
    const float nu2 = nu * kLog2e;
    const float k2 = k * kLog2e;
    float S = 0.f, D = 0.f, eprev = 0.f;
#pragma unroll
    for (int m = 0; m < 48; ++m) {
        const float t = float(m) * h;
        const float w = (m == 0) ? 0.25f * h : 0.5f * h;
        const float up = (t + eh) + el;
        const float um = (eh - t) + el;
        const float ep = __builtin_amdgcn_exp2f(nu2 * up - k2 * kCosh[m]);
        const float em = __builtin_amdgcn_exp2f(nu2 * um - k2 * kCosh[m]);
        S += w * (ep + em);
        D += w * (up * ep + um * em);
        if (ep < eprev && ep < 1e-9f * S) break;
        eprev = ep;
    }
    return D;
}

}  // namespace gsmi
