// Roundings of the transforms' kernel, of its Fourier transform and of phases
// in turns, against long double.
//
// Bounds, before any run. phi in FP64: about beta / 2 = 18 of the series'
// factors count, each with three roundings of 1.1e-16 at most (0.45e-16 rms):
// 3.3e-16 rms, twice that allowed (a rounding of t, of which I0 makes 18 times
// as much, would give 1.8e-15). 1 / phi^: nine roundings, 1.4e-16 rms, and
// exp's argument, below 2.5: 4e-16 allowed. A phase in turns: 3e-17 in all.
#include <cmath>
#include <cstdio>

#include "kaiser_bessel.hpp"

using L = long double;

namespace {

const L kPi = 3.14159265358979323846264338327950288L;

L phi(L x, int w, L beta)
{
    const L u = 2 * x / w, t = beta * beta / 4 * (1 - u * u);
    L s = 1;
    for (int k = 100; k >= 1; --k) s = 1 + s * t / (L(k) * k);
    return s * expl(-beta);
}

L inverse(L t, int w, L beta)
{
    const L r = t * w / 2, a = sqrtl(beta * beta - r * r);
    return 2 * a * expl(beta - a) / (w * (1 - expl(-2 * a)));
}

int bad = 0;

void check(const char *what, double over, double rms, double bar)
{
    std::printf("%s, oversampling %.2f: %.2e (%.1e)\n", what, over, rms, bar);
    bad += !(rms <= bar);
}

}  // namespace

int main()
{
    const int w = 16;
    for (double over : {1.9, 2.0, 2.37, 3.2}) {
        const double beta = 0.995 * 3.14159265358979323846 * w * (1.0 - 0.5 / over), e_beta = std::exp(-beta);
        L sum = 0, weight = 0;
        for (int i = 1; i < 20000; ++i) {  // by their weight in a sum
            const double x = 8.0 * (2.0 * i / 20000 - 1.0) * 0.99937;
            const L want = phi(x, w, beta), got = scarf::kaiser_bessel<66, true>(x, w, beta, e_beta);
            sum += (got - want) * (got - want);
            weight += want * want;
        }
        check("phi", over, double(sqrtl(sum / weight)), 6.6e-16);
        sum = 0;
        for (int i = 0; i < 2000; ++i) {
            const double t = 3.14159265358979323846 / over * i / 2000;
            const L want = inverse(t, w, beta), e = scarf::kaiser_bessel_inverse(t, w, beta) / want - 1;
            sum += e * e;
        }
        check("1 / phi^", over, double(sqrtl(sum / 2000)), 4e-16);
    }
    L worst = 0;
    for (int i = 0; i < 200000; ++i) {
        const double v = 1e-3 * i * 0.7548776662466927, x = 0.37 + 1e-2 * (i % 977);
        const scarf::Turns t = scarf::turns(i % 2 ? -v : v, x);
        const L want = (i % 2 ? -L(v) : L(v)) * x / (2 * kPi);
        if (fabsl(want) > 100) continue;  // beyond, long double rounds by 1e-17 itself
        L d = want - (L(t.hi) + t.lo);
        d -= rintl(d);
        worst = fmaxl(worst, fabsl(d));
        if (!(std::fabs(t.hi) <= 0.5)) ++bad;
    }
    check("turns", 0, double(worst), 3e-17);
    return bad != 0;
}
