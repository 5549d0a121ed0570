// Shortwave two-stream layer properties (sw_dif_and_source, F90:1043-1104, PIFM coefficients;
// the Rdir/Tdir clamp of src_kernels_cuda/rte_solver_kernels.cu:581-583) in FP64.
#pragma once

#include "common.h"

namespace rrtmgp_hip
{
// The layer properties.  Returns Rdif, Tdif, Rdir, Tdir (per unit incident direct flux) and the
// direct-beam transmittance Tnoscat.
__device__ __forceinline__ void sw_two_stream(double tau, double w0, double g, double mu0, double& Rdif,
                                              double& Tdif, double& Rdir, double& Tdir, double& Tnoscat)
{
    const double eps = Limits<double>::eps;
    const double gamma1 = (8. - w0 * (5. + 3. * g)) * .25;
    const double gamma2 = 3. * (w0 * (1. - g)) * .25;
    const double gamma3 = (2. - 3. * mu0 * g) * .25;
    const double gamma4 = 1. - gamma3;
    const double alpha1 = gamma1 * gamma4 + gamma2 * gamma3;
    const double alpha2 = gamma1 * gamma3 + gamma2 * gamma4;
    const double k = sqrt(fmax((gamma1 - gamma2) * (gamma1 + gamma2), Limits<double>::k_min));
    const double k_mu = k * mu0, k_gamma3 = k * gamma3, k_gamma4 = k * gamma4;
    const double e1 = exp(-tau * k);
    const double e2 = e1 * e1;
    const double RT = 1. / (k * (1. + e2) + gamma1 * (1. - e2));
    Rdif = RT * gamma2 * (1. - e2);
    Tdif = RT * 2. * k * e1;
    const double d = 1. - k_mu * k_mu;
    const double denom = (fabs(d) >= eps) ? d : eps;
    const double RT2 = w0 * RT / denom;
    Tnoscat = exp(-tau / mu0);
    double rd = RT2 * ((1. - k_mu) * (alpha2 + k_gamma3) - (1. + k_mu) * (alpha2 - k_gamma3) * e2 -
                  2. * (k_gamma3 - alpha2 * k_mu) * e1 * Tnoscat);
    double td = -RT2 * ((1. + k_mu) * (alpha1 + k_gamma4) * Tnoscat -
                   (1. - k_mu) * (alpha1 - k_gamma4) * e2 * Tnoscat -
                   2. * (k_gamma4 + alpha1 * k_mu) * e1);
    rd = fmax(fmin(rd, 1. - Tnoscat), eps);
    td = fmax(fmin(td, 1. - Tnoscat - rd), eps);
    Rdir = rd;
    Tdir = td;
}
}  // namespace rrtmgp_hip
