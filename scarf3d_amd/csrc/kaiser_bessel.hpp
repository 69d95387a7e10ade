// The compact kernel of the nonuniform transforms and its Fourier transform:
//   phi(x) = e^-beta I0(beta sqrt(1 - (2 x / w)^2)),  |x| <= w / 2 cells,
//   phi^(t) = e^-beta w sinh(a) / a,  a = sqrt(beta^2 - (w t / 2)^2), t in
//   radians per cell.
#pragma once
#include <hip/hip_runtime.h>

namespace scarf {

// I0 by its power series, all terms positive: K terms reach 1e-17 of the sum
// for beta up to 28 (K = 45) or 50 (K = 66)
template <int K>
__device__ inline double kaiser_bessel(double x, int w, double beta, double e_beta)
{
    const double u = 2.0 * x / w;
    const double t = 0.25 * beta * beta * (1.0 - u * u);
    if (!(t >= 0.0)) return 0.0;
    double s = 1.0;
#pragma unroll
    for (int k = K; k >= 1; --k) s = fma(s, t * (1.0 / (double(k) * k)), 1.0);
    return s * e_beta;
}

// 1 / phi^(t)
__device__ inline double kaiser_bessel_inverse(double t, int w, double beta)
{
    const double r = 0.5 * w * t;
    const double a = sqrt(beta * beta - r * r);
    return 2.0 * a * exp(beta - a) / (w * (1.0 - exp(-2.0 * a)));
}

}  // namespace scarf
