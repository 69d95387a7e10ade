// The compact kernel of the nonuniform transforms and its Fourier transform:
//   phi(x) = e^-beta I0(beta sqrt(1 - (2 x / w)^2)),  |x| <= w / 2 cells,
//   phi^(t) = e^-beta w sinh(a) / a,  a = sqrt(beta^2 - (w t / 2)^2), t in
//   radians per cell.
#pragma once
#include <hip/hip_runtime.h>

namespace scarf {

// I0(2 sqrt t) by its power series, all terms positive: K terms reach 1e-17 of
// the sum for beta up to 28 (K = 45) or 50 (K = 66). It answers a relative
// error of t with up to beta / 2 times as large a one, so for FP64 fields what
// the roundings of t leave out is put back by the derivative, I0 sqrt(1 / t)
// from t = 1 on (Exact; w a power of two, so that u is exact): 1.2e-15 ->
// 5e-16 of phi.
template <int K, bool Exact = false>
__host__ __device__ inline double kaiser_bessel(double x, int w, double beta, double e_beta)
{
#pragma clang fp contract(off)
    const double u = 2.0 * x / w, half = 0.5 * beta, c = half * half;
    const double e = fma(-u, u, 1.0), t = c * e;
    if (!(t >= 0.0)) return 0.0;
    double s = 1.0;
#pragma unroll
    for (int k = K; k >= 1; --k) s = fma(s, t * (1.0 / (double(k) * k)), 1.0);
    if constexpr (Exact) {
        const double rest = fma(c, e, -t) + (fma(half, half, -c) * e + c * fma(-u, u, 1.0 - e));
        s = fma(s, rest / sqrt(t > 1.0 ? t : 1.0), s);
    }
    return s * e_beta;
}

// 1 / phi^(t); beta - a by its product with beta + a, since beta and a are some
// 40 and their roundings 30 times exp's own
__host__ __device__ inline double kaiser_bessel_inverse(double t, int w, double beta)
{
    const double r = 0.5 * w * t;
    const double a = sqrt(beta * beta - r * r);
    return 2.0 * a * exp(r * r / (beta + a)) / (w * (1.0 - exp(-2.0 * a)));
}

// w x in turns modulo 1, to the last bit of the part that is left: hi + lo
struct Turns {
    double hi, lo;
};
__host__ __device__ inline Turns turns(double w, double x)
{
#pragma clang fp contract(off)
    constexpr double inv = 0.15915494309189533577, inv_lo = -9.839338337591243e-18;  // of 1 / (2 pi)
    const double p = w * x, h = p * inv;
    return Turns{h - rint(h), fma(p, inv, -h) + (fma(w, x, -p) * inv + p * inv_lo)};
}

}  // namespace scarf
