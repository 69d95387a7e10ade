// The dense transform of short lines in float against an FP64 transform on the
// host: 2-norm error over 2-norm of the result.
//
// Bounds, before any run. A rounding to FP32 is 2.4e-8 rms. A line's products sum
// in chains of 4 terms (up to 64) or 8 (up to 128 or 288): 2.4e-8 sqrt(c / 2), 3.4e-8 or
// 4.8e-8; the folded inputs, the matrices, the twiddles and the result round once
// each, 4.8e-8. Over three axes 1.02e-7 and 1.18e-7; a sixth more allowed. (With
// chains of 16, totals and combinations in FP32: 1.6e-7.)
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include <hip/hip_runtime.h>

#include "fim_dft.hpp"

using C = std::complex<double>;

namespace {

int bad = 0;

void need(hipError_t e, const char *what)
{
    if (e == hipSuccess) return;
    std::printf("%s: %s\n", what, hipGetErrorString(e));
    std::exit(2);
}

// lines of n values `stride` apart: first values base(l), l < lines
template <class Base>
void host_lines(std::vector<C> &v, int n, long stride, long lines, const Base &base)
{
    std::vector<C> w(n), in(n);
    for (int q = 0; q < n; ++q) w[q] = std::polar(1.0, 2.0 * M_PI * q / n);
    for (long l = 0; l < lines; ++l) {
        C *p = v.data() + base(l);
        for (int q = 0; q < n; ++q) in[q] = p[q * stride];
        for (int k = 0; k < n; ++k) {
            C s = 0;
            for (int q = 0; q < n; ++q) s += w[long(k) * q % n] * in[q];
            p[k * stride] = s;
        }
    }
}

void check(int n1, int n2, int n3, double bar)
{
    std::printf("[case] %d x %d x %d\n", n1, n2, n3);
    std::fflush(stdout);
    const int h = n1 / 2 + 1;
    const size_t half = size_t(h) * n2 * n3, total = size_t(n1) * n2 * n3;
    std::vector<std::complex<float>> s(half);
    std::vector<C> t(half);
    unsigned r = 7;
    auto next = [&] {
        r = r * 1664525u + 1013904223u;
        return float((r >> 8) / 16777216.0 - 0.5);
    };
    for (size_t i = 0; i < half; ++i) {
        s[i] = {next(), next()};
        t[i] = C(s[i].real(), s[i].imag());
    }
    if (!scarf::fim_dft::chosen<float>(n1, n2, n3)) ++bad, std::printf("not a dense transform\n");
    void *ds = nullptr, *tables = nullptr;
    float *dr = nullptr;
    double *part = nullptr;
    need(hipMalloc(&ds, half * 8), "hipMalloc");
    need(hipMalloc(reinterpret_cast<void **>(&dr), total * 4), "hipMalloc");
    need(hipMalloc(&tables, scarf::fim_dft::table_bytes<float>(n1, n2, n3)), "hipMalloc");
    need(hipMalloc(reinterpret_cast<void **>(&part), 24 * scarf::fim_dft::parts<float>(n1, n2, n3)), "hipMalloc");
    need(hipMemcpy(ds, s.data(), half * 8, hipMemcpyHostToDevice), "hipMemcpy");
    need(scarf::fim_dft::make_tables<float>(tables, n1, n2, n3, nullptr), "make_tables");
    need(scarf::fim_dft::run<float>(ds, dr, {}, tables, n1, n2, n3, 1.f, part, nullptr), "run");
    std::vector<float> got(total);
    need(hipMemcpy(got.data(), dr, total * 4, hipMemcpyDeviceToHost), "hipMemcpy");
    const long plane = long(h) * n2;
    if (n3 > 1) host_lines(t, n3, plane, plane, [](long l) { return l; });
    host_lines(t, n2, h, long(h) * n3, [&](long l) { return l / h * plane + l % h; });
    std::vector<C> w(n1);
    for (int q = 0; q < n1; ++q) w[q] = std::polar(1.0, 2.0 * M_PI * q / n1);
    double err = 0, norm = 0;
    for (long l = 0; l < long(n2) * n3; ++l)
        for (int i = 0; i < n1; ++i) {
            const C *p = t.data() + l * h;
            double v = p[0].real() + (i % 2 ? -1.0 : 1.0) * p[h - 1].real();
            for (int k = 1; k < h - 1; ++k) v += 2.0 * (w[long(k) * i % n1] * p[k]).real();
            const double d = got[l * n1 + i] - v;
            err += d * d;
            norm += v * v;
        }
    const double e = std::sqrt(err / norm);
    std::printf("  %.2e (%.2e)\n", e, bar);
    std::fflush(stdout);
    bad += !(e <= bar);
    (void)hipFree(ds);
    (void)hipFree(dr);
    (void)hipFree(tables);
    (void)hipFree(part);
}

}  // namespace

int main()
{
    const double four = 1.2e-7, eight = 1.4e-7;
    check(62, 58, 64, four);
    check(2, 38, 46, four);
    check(64, 62, 1, four);
    check(66, 70, 122, eight);
    check(128, 126, 94, eight);
    check(128, 62, 40, eight);
    check(256, 40, 38, eight);  // one axis with a large prime factor: up to 288
    check(38, 288, 130, eight);
    check(258, 128, 1, eight);
    std::printf("%d bad\n", bad);
    return bad != 0;
}
