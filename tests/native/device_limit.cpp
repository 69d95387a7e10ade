// Calls at SCARF_DEVICE_MEMORY_LIMIT, through the C interface. A limit that
// holds what a call computes from and its direct sum's tables (the formulas
// below) has to be enough, for the first call and for every later one, whatever
// workspaces earlier calls without a limit left behind; and what the library
// holds after a call is within the limit.
//   usage: device_limit     prints "ok" lines, "bad" lines, then "<n> bad"
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "device_budget.hpp"
#include "scarf3d.h"
#include "scarf3d_srm.h"

namespace {

constexpr bool kDouble = sizeof(real) == sizeof(double);
int bad = 0;

void limit(size_t bytes)
{
    if (bytes) setenv("SCARF_DEVICE_MEMORY_LIMIT", std::to_string(bytes).c_str(), 1);
    else unsetenv("SCARF_DEVICE_MEMORY_LIMIT");
}

struct Grid {
    int n[3];
    real ds, cl[3];
    int acf, method, nharm;
    int kernel = SCARF_KERNEL_AUTO;
    size_t points() const { return size_t(n[0]) * n[1] * n[2]; }
};

std::string grid(const Grid &g, int seed, std::vector<real> &field)
{
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = g.method;
    o.hurst = real(0.3);
    const int fs[3] = {1, 1, 1};
    field.assign(g.points(), real(0));
    real stats[8];
    scarf_cart_initialize(3, fs, g.n, g.ds, g.acf, g.cl, real(0.05), &o);
    scarf_set_nharm(g.nharm);
    scarf_set_kernel(g.kernel);
    scarf_execute(seed, field.data(), stats);
    const std::string e = scarf_last_error();
    scarf_finalize();
    return e;
}

std::string points(const std::vector<real> (&p)[3], int nharm, int method, int seed, std::vector<real> &field,
                   int kernel = SCARF_KERNEL_AUTO)
{
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = method;
    o.hurst = real(0.3);
    const real cl[3] = {300, 250, 200};
    const int n = int(p[0].size());
    field.assign(n, real(0));
    real stats[8];
    scarf_nocart_initialize(3, n, p[0].data(), p[1].data(), p[2].data(), real(40), 0, cl, real(0.05), &o);
    scarf_set_nharm(nharm);
    scarf_set_kernel(kernel);
    scarf_execute(seed, field.data(), stats);
    const std::string e = scarf_last_error();
    scarf_finalize();
    return e;
}

void say(const char *what, const std::string &err, size_t lim, bool same = true)
{
    const size_t held = scarf::device_budget().held();
    const bool fine = err.empty() && same && (lim == 0 || held <= lim);
    bad += !fine;
    std::printf("%s %s: limit %zu, held %zu%s%s%s\n", fine ? "ok" : "bad", what, lim, held, err.empty() ? "" : ", ",
                err.c_str(), same ? "" : ", another field");
    std::fflush(stdout);
}

double far(const std::vector<real> &a, const std::vector<real> &b)
{
    double d = 0, s = 0;
    for (size_t i = 0; i < a.size(); ++i) {
        d = std::max(d, std::fabs(double(a[i]) - b[i]));
        s = std::max(s, std::fabs(double(b[i])));
    }
    return d / s;
}
constexpr double kNear = kDouble ? 1e-10 : 1e-4;

// the record and the direct sums' tables and partials
size_t padded(int nharm) { return size_t((nharm + 63) / 64 * 64); }
size_t record(int nharm) { return 5 * padded(nharm) * sizeof(double); }
size_t direct_grid(const Grid &g)
{
    const size_t np = padded(g.nharm), lines = size_t(g.n[1]) * g.n[2];
    return np * (g.n[0] + g.n[1] + g.n[2]) * (kDouble ? 8 : 4) + np * sizeof(float) +
           3 * sizeof(double) * ((g.n[0] + 63) / 64) * ((lines + 63) / 64);
}

}  // namespace

int main()
{
    std::vector<real> a, b, c, d;
    const Grid g{{40, 30, 20}, 50, {300, 250, 200}, 0, 1, 2000};
    const size_t field = g.points() * sizeof(real);
    const size_t need = field + record(g.nharm) + direct_grid(g);

    // a grid: twice at the limit, after a call without one, and again
    limit(need);
    std::string e = grid(g, 1, a);
    say("grid, first call", e, need);
    e = grid(g, 1, b);
    say("grid, second call", e, need, a == b);
    limit(0);
    e = grid(g, 1, c);
    say("grid, no limit", e, 0, far(c, a) <= kNear);
    limit(need);
    e = grid(g, 1, b);
    say("grid, third call", e, need, a == b);
    limit(0);
    Grid direct = g;
    direct.kernel = kDouble ? SCARF_KERNEL_DIRECT_F64 : SCARF_KERNEL_DIRECT_F32;
    e = grid(direct, 1, b);
    say("grid, direct sum", e, 0, a == b);  // what the limit left room for

    // a point list, with the grid's field buffer and record still held
    std::vector<real> p[3];
    const int n = 20000, nharm = 1900;
    for (int q = 0; q < 3; ++q)
        for (int i = 0; i < n; ++i) p[q].push_back(real((i * (7919LL + 104 * q) % 20011) * (0.1 - 0.02 * q)));
    const size_t list = std::max(field, n * sizeof(real)) + record(g.nharm) + 3 * sizeof(double) * size_t(n) +
                        3 * sizeof(double) * ((n + 255) / 256);
    limit(0);
    e = points(p, nharm, 1, 3, c);
    say("points, no limit", e, 0);
    // the raw coordinates go by way of a workspace
    const size_t raw = 3 * sizeof(real) * size_t(n);
    limit(list + raw);
    e = points(p, nharm, 1, 3, a);
    say("points, at the limit", e, list + raw, far(a, c) <= kNear);
    e = points(p, nharm, 1, 3, b);
    say("points, again", e, list + raw, a == b);

    // FIM, its tables in the way: the limit is found from the refusals
    const Grid f{{33, 37, 45}, 50, {300, 250, 200}, 0, 0, 1};  // a factor above 13 in an internal axis
    limit(0);
    e = grid(f, 5, c);
    say("fim, no limit", e, 0);
    size_t lim = 1;
    for (int q = 0; q < 20; ++q) {
        limit(lim);
        e = grid(f, 5, a);
        const size_t at = e.find("would need ");
        if (e.empty() || at == std::string::npos) break;
        lim = size_t(std::atoll(e.c_str() + at + 11));
    }
    say("fim, at the limit", e, lim, far(a, c) <= kNear);
    limit(0);
    e = grid(g, 1, d);
    e = e.empty() ? grid(f, 5, b) : e;
    say("fim after a spectral field, no limit", e, 0, b == c);
    limit(lim);
    e = grid(f, 5, b);
    say("fim after a spectral field", e, lim, a == b);
    e = points(p, nharm, 0, 5, b);
    if (!e.empty() && e.find("SCARF_DEVICE_MEMORY_LIMIT") == std::string::npos) say("fim points", e, lim);
    limit(lim + 3 * sizeof(double) * size_t(n) + raw);
    e = points(p, nharm, 0, 5, b);
    say("fim points", e, lim + 3 * sizeof(double) * size_t(n) + raw);

    // an ensemble, whose own buffers the limit does not count
    std::vector<scarf_member> members(5);
    std::vector<real *> fields;
    for (size_t m = 0; m < members.size(); ++m) {
        scarf_member &s = members[m];
        std::memset(&s, 0, sizeof s);
        s.nd = 3;
        for (int q = 0; q < 3; ++q) {
            s.fs[q] = 1;
            s.fe[q] = g.n[q] + int(m);
            s.cl[q] = g.cl[q];
        }
        s.ds = g.ds;
        s.hurst = real(0.3);
        s.sigma = real(0.05);
        s.nharm = 1500;
        s.seed = int(m) + 1;
        void *ptr = nullptr;
        if (hipMalloc(&ptr, size_t(s.fe[0]) * s.fe[1] * s.fe[2] * sizeof(real)) != hipSuccess) return 2;
        fields.push_back(static_cast<real *>(ptr));
    }
    std::vector<real> stats(8 * members.size());
    lim = scarf::device_budget().held();
    for (int q = 0; q < 2; ++q) {
        limit(q == 0 ? lim : 0);
        const int rc = scarf_ensemble_execute(int(members.size()), members.data(), fields.data(), stats.data(), 0);
        say(q == 0 ? "ensemble at the limit" : "ensemble", rc == 0 ? "" : scarf_last_error(), q == 0 ? lim : 0);
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
