// Kernel values of the Duffy table builds (duffy.hip, duffy_tensor.hip).
#pragma once

#include <cmath>

#include "internal.h"

namespace vl1 {

// Kernel values, sumpy conventions (expression times global scaling):
// Laplace 2D -log(r)/(2 pi), 3D 1/(4 pi r); Helmholtz 2D (i/4) H0^(1)(k r)
// = (-Y0(kr) + i J0(kr)) / 4, 3D e^{ikr}/(4 pi r).  Axis derivatives of
// Laplace (da = component of d = target - source on the derivative axis):
// target dG/dd_a = 2D -da/(2 pi r^2), 3D -da/(4 pi r^3); source = minus.
// Axis derivatives of Helmholtz: G'(r) da / r with G' = 2D -(ik/4) H1^(1)(kr)
// = (k/4)(Y1(kr) - i J1(kr)), 3D e^{ikr}(ikr - 1)/(4 pi r^2).  Radial terms
// of the Helmholtz split: r^p and r^p log r, no scaling constant (the
// exponent p travels in the k slot).
__host__ __device__ constexpr bool kind_is_complex(int kind) {
  return kind == VL1_KERNEL_HELMHOLTZ || kind == VL1_KERNEL_HELMHOLTZ_TARGET_DERIV ||
         kind == VL1_KERNEL_HELMHOLTZ_SOURCE_DERIV;
}
__host__ __device__ constexpr bool kind_is_power_deriv(int kind) {
  return kind == VL1_KERNEL_POWER_TARGET_DERIV || kind == VL1_KERNEL_POWER_SOURCE_DERIV ||
         kind == VL1_KERNEL_POWER_LOG_TARGET_DERIV || kind == VL1_KERNEL_POWER_LOG_SOURCE_DERIV;
}
__host__ __device__ constexpr bool kind_is_deriv(int kind) {
  return kind == VL1_KERNEL_LAPLACE_TARGET_DERIV || kind == VL1_KERNEL_LAPLACE_SOURCE_DERIV ||
         kind == VL1_KERNEL_HELMHOLTZ_TARGET_DERIV || kind == VL1_KERNEL_HELMHOLTZ_SOURCE_DERIV ||
         kind_is_power_deriv(kind);
}
template <int DIM, int KIND>
__device__ inline void kernel_value(double r2, double da, double k, double& re, double& im) {
  if (KIND == VL1_KERNEL_LAPLACE_TARGET_DERIV || KIND == VL1_KERNEL_LAPLACE_SOURCE_DERIV) {
    constexpr double sgn = KIND == VL1_KERNEL_LAPLACE_TARGET_DERIV ? -1.0 : 1.0;
    if (DIM == 2) {
      re = sgn * 0.5 / M_PI * da / r2;
    } else {
      const double ir = rsqrt(r2);
      re = sgn * 0.25 / M_PI * da * ir * ir * ir;
    }
    im = 0.0;
  } else if (KIND == VL1_KERNEL_HELMHOLTZ_TARGET_DERIV || KIND == VL1_KERNEL_HELMHOLTZ_SOURCE_DERIV) {
    constexpr double sgn = KIND == VL1_KERNEL_HELMHOLTZ_TARGET_DERIV ? 1.0 : -1.0;
    const double ir = rsqrt(r2);
    const double r = r2 * ir;
    const double kr = k * r;
    if (DIM == 2) {
      const double f = sgn * 0.25 * k * da * ir;
      re = f * y1(kr);
      im = -f * j1(kr);
    } else {
      double sn, cs;
      sincos(kr, &sn, &cs);
      const double f = sgn * 0.25 / M_PI * da * ir * ir * ir;
      re = f * (-cs - kr * sn);
      im = f * (kr * cs - sn);
    }
  } else if (KIND == VL1_KERNEL_CONSTANT) {
    re = 1.0;
    im = 0.0;
  } else if (kind_is_power_deriv(KIND)) {
    // d_a |d|^(p-2) times p, or times (p log|d| + 1) with the log (k carries p)
    constexpr bool tgt =
        KIND == VL1_KERNEL_POWER_TARGET_DERIV || KIND == VL1_KERNEL_POWER_LOG_TARGET_DERIV;
    constexpr bool lg =
        KIND == VL1_KERNEL_POWER_LOG_TARGET_DERIV || KIND == VL1_KERNEL_POWER_LOG_SOURCE_DERIV;
    const double base = da * pow(r2, 0.5 * k - 1.0);
    re = (tgt ? 1.0 : -1.0) * base * (lg ? fma(0.5 * k, log(r2), 1.0) : k);
    im = 0.0;
  } else if (KIND == VL1_KERNEL_POWER || KIND == VL1_KERNEL_POWER_LOG) {
    // |d|^p (k carries p for these kinds), times log|d| for POWER_LOG
    re = pow(r2, 0.5 * k);
    if (KIND == VL1_KERNEL_POWER_LOG) re *= 0.5 * log(r2);
    im = 0.0;
  } else if (KIND == VL1_KERNEL_LAPLACE) {
    if (DIM == 2) {
      re = -0.25 / M_PI * log(r2);
    } else {
      re = 0.25 / M_PI * rsqrt(r2);
    }
    im = 0.0;
  } else if (DIM == 2) {
    const double kr = k * sqrt(r2);
    re = -0.25 * y0(kr);
    im = 0.25 * j0(kr);
  } else {
    const double ir = rsqrt(r2);
    double sn, cs;
    sincos(k * (r2 * ir), &sn, &cs);
    re = 0.25 / M_PI * cs * ir;
    im = 0.25 / M_PI * sn * ir;
  }
}

}  // namespace vl1
